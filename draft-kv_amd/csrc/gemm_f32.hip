// float32 projections of the model forwards on the float32 matrix cores:
// out (+)= x[M][K] . w (+ bias), w[K][N] (layout 0) or w[N][K] (layout 1).
// Reference: the `x @ W` products of model.py:113-133, gpt2.py:191-213,
// llama.py:187-225.
//
// Arithmetic (the same for every M and launch shape, so a verify row equals
// the one-token decode row bit for bit): K is cut into chunks fixed by
// (N, K); per chunk an output is one chain of v_mfma_f32_16x16x4_f32 over the
// chunk's 16-k groups (step e of a group takes k = 4 j + e, j = 0..3), the
// chunk sums are added in chunk order, then the bias.
//
// Operands go from memory straight to registers: lane (col, j) of a wave
// loads x[row col][4 j .. + 3] of a group, the k-slots of four MFMA steps in
// one 16-byte load. Layout 1 does the same with a 16-row fragment of w. In
// layout 0 the lane loads the NW consecutive columns NW col .. of row
// 4 j + e, and component f is the A operand of subtile f, whose rows are then
// the columns NW i + f. A float32 MFMA takes 32 cycles for 64 FLOP a cycle
// and SIMD, so even a 16 x 16 tile needs only 32 bytes a cycle and CU of w:
// no LDS staging, at decode sizes w streams from HBM, at prefill sizes both
// operands come from L1 and L2.
#include <algorithm>

#include "dkv_common.h"

namespace dkv {

typedef float ff32x4_t __attribute__((ext_vector_type(4)));

struct GemmF32Args {
    const float* x;
    const float* w;
    const void* bias;
    int bias_dtype;
    float* out;
    int M, N, K, KC, S;   // S chunks of KC (a multiple of 16; the last one may be short)
    int accumulate;
    int vec_out;          // rows of out are 16-byte aligned
};

__device__ __forceinline__ float gemm_bias(const GemmF32Args& a, int n) {
    return a.bias ? load_elem(a.bias, n, a.bias_dtype) : 0.0f;
}

// outputs out[m][n .. n + 3] += t (+ bias), up to column N - 1
__device__ __forceinline__ void gemm_store4(const GemmF32Args& a, int m, int n, ff32x4_t t) {
    float* p = a.out + (int64_t)m * a.N + n;
    if (a.vec_out && n + 3 < a.N) {
        float4 v = make_float4(t[0] + gemm_bias(a, n), t[1] + gemm_bias(a, n + 1), t[2] + gemm_bias(a, n + 2),
                               t[3] + gemm_bias(a, n + 3));
        if (a.accumulate) {
            const float4 h = *reinterpret_cast<const float4*>(p);
            v = make_float4(h.x + v.x, h.y + v.y, h.z + v.z, h.w + v.w);
        }
        *reinterpret_cast<float4*>(p) = v;
        return;
    }
#pragma unroll
    for (int e = 0; e < 4; ++e)
        if (n + e < a.N) {
            const float v = t[e] + gemm_bias(a, n + e);
            p[e] = a.accumulate ? p[e] + v : v;
        }
}

// A wave's tile: NW 16-column fragments of N by MB 16-row fragments of M.
// SPLIT: the workgroup's S waves take one chunk each of the same tile, and
// the sums meet in LDS; else its four waves own a 2 x 2 block of tiles (four
// tiles along N when MB * 16 covers M) and walk the chunks in order. VEC:
// K % 4 == 0 and aligned rows, so the loads are vectors.
template <int WL, int NW, int MB, bool SPLIT, bool VEC>
__global__ void __launch_bounds__(SPLIT ? 1024 : 256) gemm_f32_kernel(GemmF32Args a, int two_by_two) {
#pragma clang fp contract(off)
    constexpr int U = NW * MB >= 8 ? 1 : NW * MB >= 4 ? 2 : 4;   // 16-k groups per register set
    extern __shared__ __align__(16) float red[];                 // SPLIT: [S][NW * MB][64 lanes][4]
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / WAVE), lane = threadIdx.x % WAVE;
    const int col = lane % 16, j = lane / 16;
    int tn = blockIdx.x, tm = blockIdx.y;
    if (!SPLIT) {
        tn = two_by_two ? 2 * tn + (wave & 1) : 4 * tn + wave;
        tm = two_by_two ? 2 * tm + (wave >> 1) : tm;
    }
    const int n0 = tn * 16 * NW, m0 = tm * 16 * MB;
    if (!SPLIT && (n0 >= a.N || m0 >= a.M)) return;
    const int K = a.K, N = a.N;
    // rows past M and columns past N reread the last one; their products are never stored
    const float* xp[MB];
#pragma unroll
    for (int b = 0; b < MB; ++b) xp[b] = a.x + (int64_t)min(m0 + 16 * b + col, a.M - 1) * K;
    const float* wp[WL ? NW : 1];
    if constexpr (WL) {
#pragma unroll
        for (int f = 0; f < NW; ++f) wp[f] = a.w + (int64_t)min(n0 + 16 * f + col, N - 1) * K;
    } else {
        wp[0] = a.w + min(n0 + NW * col, N - NW);   // N >= NW, and N % NW == 0 where NW > 1
    }

    struct Regs {
        float w[U][NW][4];   // [group][fragment][step]
        float x[U][MB][4];
    };
    // groups g0 .. g0 + U - 1 from k; groups at or past `kend` read group kend - 16 again (and are not multiplied).
    // FULL: the 16 k of every group lie below K
    auto load = [&](Regs& r, int k, int kend, bool full) {
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int kg = min(k + 16 * u, kend - 16 + (-kend & 15)) + 4 * j;
            if (VEC && (full || kg + 4 <= K)) {
#pragma unroll
                for (int b = 0; b < MB; ++b) {
                    const float4 v = *reinterpret_cast<const float4*>(xp[b] + kg);
                    r.x[u][b][0] = v.x, r.x[u][b][1] = v.y, r.x[u][b][2] = v.z, r.x[u][b][3] = v.w;
                }
                if constexpr (WL) {
#pragma unroll
                    for (int f = 0; f < NW; ++f) {
                        const float4 v = *reinterpret_cast<const float4*>(wp[f] + kg);
                        r.w[u][f][0] = v.x, r.w[u][f][1] = v.y, r.w[u][f][2] = v.z, r.w[u][f][3] = v.w;
                    }
                } else {
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        const float* p = wp[0] + (int64_t)(kg + e) * N;
                        if constexpr (NW == 4) {
                            const float4 v = *reinterpret_cast<const float4*>(p);
                            r.w[u][0][e] = v.x, r.w[u][1][e] = v.y, r.w[u][2][e] = v.z, r.w[u][3][e] = v.w;
                        } else if constexpr (NW == 2) {
                            const float2 v = *reinterpret_cast<const float2*>(p);
                            r.w[u][0][e] = v.x, r.w[u][1][e] = v.y;
                        } else {
                            r.w[u][0][e] = *p;
                        }
                    }
                }
            } else {
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const bool in = kg + e < K;
#pragma unroll
                    for (int b = 0; b < MB; ++b) r.x[u][b][e] = in ? xp[b][kg + e] : 0.0f;
                    if constexpr (WL) {
#pragma unroll
                        for (int f = 0; f < NW; ++f) r.w[u][f][e] = in ? wp[f][kg + e] : 0.0f;
                    } else {
#pragma unroll
                        for (int f = 0; f < NW; ++f) r.w[u][f][e] = in ? wp[0][(int64_t)(kg + e) * N + f] : 0.0f;
                    }
                }
            }
        }
    };
    ff32x4_t acc[NW][MB], tot[SPLIT ? 1 : NW][SPLIT ? 1 : MB];
    auto clear = [&]() {
#pragma unroll
        for (int f = 0; f < NW; ++f)
#pragma unroll
            for (int b = 0; b < MB; ++b) acc[f][b] = ff32x4_t{0.f, 0.f, 0.f, 0.f};
    };
    auto mul = [&](const Regs& r, int k, int kend) {
#pragma unroll
        for (int u = 0; u < U; ++u)
            if (U == 1 || k + 16 * u < kend) {
#pragma unroll
                for (int e = 0; e < 4; ++e)
#pragma unroll
                    for (int f = 0; f < NW; ++f)
#pragma unroll
                        for (int b = 0; b < MB; ++b)
                            acc[f][b] = __builtin_amdgcn_mfma_f32_16x16x4f32(r.w[u][f][e], r.x[u][b][e], acc[f][b], 0, 0, 0);
            }
    };
    const int c0 = SPLIT ? wave : 0, c1 = SPLIT ? wave + 1 : a.S;
    for (int c = c0; c < c1; ++c) {
        const int kb = c * a.KC, kend = min(kb + a.KC, K);
        const bool full = kend % 16 == 0;
        clear();
        Regs r0, r1;
        load(r0, kb, kend, full);
        for (int k = kb; k < kend; k += 32 * U) {
            if (k + 16 * U < kend) load(r1, k + 16 * U, kend, full);
            mul(r0, k, kend);
            if (k + 16 * U >= kend) break;
            if (k + 32 * U < kend) load(r0, k + 32 * U, kend, full);
            mul(r1, k + 16 * U, kend);
        }
        if constexpr (!SPLIT) {
#pragma unroll
            for (int f = 0; f < NW; ++f)
#pragma unroll
                for (int b = 0; b < MB; ++b) {
                    if (c == 0) tot[f][b] = acc[f][b];
                    else
#pragma unroll
                        for (int e = 0; e < 4; ++e) tot[f][b][e] = tot[f][b][e] + acc[f][b][e];
                }
        }
    }
    if constexpr (SPLIT) {
#pragma unroll
        for (int f = 0; f < NW; ++f)
#pragma unroll
            for (int b = 0; b < MB; ++b)
                *reinterpret_cast<ff32x4_t*>(red + (((wave * NW + f) * MB + b) * WAVE + lane) * 4) = acc[f][b];
        __syncthreads();
        // wave w sums and stores the subtiles w, w + S, ... (layout 0 with NW > 1: row r of every f together)
        for (int i = wave; i < NW * MB; i += a.S) {
            const int f = i / MB, b = i % MB, m = m0 + 16 * b + col;
            ff32x4_t t = *reinterpret_cast<const ff32x4_t*>(red + ((f * MB + b) * WAVE + lane) * 4);
            for (int c = 1; c < a.S; ++c) {
                const ff32x4_t v = *reinterpret_cast<const ff32x4_t*>(red + (((c * NW + f) * MB + b) * WAVE + lane) * 4);
#pragma unroll
                for (int e = 0; e < 4; ++e) t[e] = t[e] + v[e];
            }
            if (m >= a.M) continue;
            if constexpr (WL == 1 || NW == 1) {
                gemm_store4(a, m, n0 + 16 * f + 4 * j, t);
            } else {
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const int n = n0 + NW * (4 * j + e) + f;
                    if (n < N) {
                        const float v = t[e] + gemm_bias(a, n);
                        float* p = a.out + (int64_t)m * N + n;
                        *p = a.accumulate ? *p + v : v;
                    }
                }
            }
        }
    } else {
#pragma unroll
        for (int b = 0; b < MB; ++b) {
            const int m = m0 + 16 * b + col;
            if (m >= a.M) continue;
            if constexpr (WL == 1 || NW == 1) {
#pragma unroll
                for (int f = 0; f < NW; ++f) gemm_store4(a, m, n0 + 16 * f + 4 * j, tot[f][b]);
            } else {   // the lane holds 4 NW consecutive columns: n0 + NW (4 j + e) + f
                constexpr int Q = NW;
#pragma unroll
                for (int v = 0; v < Q; ++v) {
                    ff32x4_t t;
#pragma unroll
                    for (int e = 0; e < 4; ++e) t[e] = tot[(4 * v + e) % NW][b][(4 * v + e) / NW];
                    gemm_store4(a, m, n0 + 4 * NW * j + 4 * v, t);
                }
            }
        }
    }
}

// K chunks, a function of (N, K) only: enough for about 1024 waves (one per
// SIMD) of 16 columns, at most 16, each at least 64 long
struct ChunksF32 {
    int KC, S;
};
static ChunksF32 gemm_f32_chunks(int N, int K) {
    const int frags = (N + 15) / 16;
    const int s = std::max(1, std::min(std::min(16, K / 64), (1024 + frags - 1) / frags));
    ChunksF32 c;
    c.KC = ((K + s - 1) / s + 15) / 16 * 16;
    c.S = (K + c.KC - 1) / c.KC;
    return c;
}

template <int WL, int NW, int MB, bool SPLIT, bool VEC>
static int launch_f32(const GemmF32Args& a, bool two_by_two, hipStream_t st) {
    const int64_t tn = (a.N + 16 * NW - 1) / (16 * NW), tm = (a.M + 16 * MB - 1) / (16 * MB);
    const int64_t gx = SPLIT ? tn : two_by_two ? (tn + 1) / 2 : (tn + 3) / 4;
    const int64_t gy = !SPLIT && two_by_two ? (tm + 1) / 2 : tm;
    const size_t lds = SPLIT ? sizeof(float) * 256 * (size_t)a.S * NW * MB : 0;
    hipLaunchKernelGGL((gemm_f32_kernel<WL, NW, MB, SPLIT, VEC>), dim3((unsigned)gx, (unsigned)gy),
                       dim3(SPLIT ? 64 * a.S : 256), lds, st, a, (int)two_by_two);
    return check_launch("dkv_gemm_f32");
}

template <int WL>
static int launch_f32_wl(const GemmF32Args& a, bool vec, bool wide, hipStream_t st) {
    const bool split = a.S > 1;
    if (!vec) return split ? launch_f32<WL, 1, 1, true, false>(a, false, st) : launch_f32<WL, 1, 1, false, false>(a, false, st);
    // few rows: one fragment of w per wave, every row beside it, w read once
    if (a.M <= 16) return split ? launch_f32<WL, 1, 1, true, true>(a, false, st) : launch_f32<WL, 1, 1, false, true>(a, false, st);
    if (a.M <= 32) return split ? launch_f32<WL, 1, 2, true, true>(a, false, st) : launch_f32<WL, 1, 2, false, true>(a, false, st);
    if (a.M <= 64) return split ? launch_f32<WL, 1, 4, true, true>(a, false, st) : launch_f32<WL, 1, 4, false, true>(a, false, st);
    const int64_t w44 = (int64_t)((a.N + 63) / 64) * ((a.M + 63) / 64), w22 = (int64_t)((a.N + 31) / 32) * ((a.M + 31) / 32);
    if (w44 >= 1024 && wide) return launch_f32<WL, 4, 4, false, true>(a, true, st);
    if (w22 >= 512 || !split) {
        if (wide) return launch_f32<WL, 2, 2, false, true>(a, true, st);
        return launch_f32<WL, 1, 4, false, true>(a, false, st);
    }
    if (wide) return launch_f32<WL, 2, 2, true, true>(a, false, st);
    return launch_f32<WL, 1, 4, true, true>(a, false, st);
}

}  // namespace dkv

using namespace dkv;

extern "C" int dkv_gemm_f32(const float* x, const float* w, int32_t w_layout, int32_t M, int32_t N, int32_t K,
                            const void* bias, int32_t bias_dtype, float* out, int32_t accumulate,
                            dkv_stream_t stream) {
    DKV_REQUIRE(x && w && out && N > 0 && K > 0 && (w_layout == 0 || w_layout == 1), "dkv_gemm_f32: bad arguments");
    DKV_REQUIRE(!bias || bias_dtype == DKV_F32 || bias_dtype == DKV_BF16, "dkv_gemm_f32: bad bias dtype");
    DKV_REQUIRE(M <= 65535 * 16, "dkv_gemm_f32: too many rows for one launch");
    if (M <= 0) return DKV_OK;
    const ChunksF32 c = gemm_f32_chunks(N, K);
    auto aligned = [](const void* p) { return reinterpret_cast<uintptr_t>(p) % 16 == 0; };
    GemmF32Args a;
    a.x = x, a.w = w, a.bias = bias, a.bias_dtype = bias_dtype, a.out = out;
    a.M = M, a.N = N, a.K = K, a.KC = c.KC, a.S = c.S, a.accumulate = accumulate;
    a.vec_out = N % 4 == 0 && aligned(out);
    const bool vec = K % 4 == 0 && aligned(x) && (w_layout == 0 || aligned(w));
    const bool wide = w_layout == 1 || (N % 4 == 0 && aligned(w));   // layout 0 reads vectors along N
    return w_layout == 1 ? launch_f32_wl<1>(a, vec, wide, as_stream(stream))
                         : launch_f32_wl<0>(a, vec, wide, as_stream(stream));
}

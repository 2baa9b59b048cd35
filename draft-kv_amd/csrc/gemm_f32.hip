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
// at decode sizes w streams from HBM into registers with no LDS staging;
// prompts share operands through LDS (gemm_f32_lds_kernel).
//
// Against one thread per output with both operands in LDS: the 121 products of
// a SmolLM2-135M decode step 36.8 -> 6.7 us on average (SwiGLU included), the
// 25 of a 1000-token distilgpt2 prompt 443 -> 108 us (its head at 100 TFLOP/s
// of the 154 a library product reaches).
#include <algorithm>

#include "dkv_common.h"

namespace dkv {

typedef float ff32x4_t __attribute__((ext_vector_type(4)));
// loads of 4-byte aligned rows (any K, any caller's pointer)
typedef float ff32x4u_t __attribute__((ext_vector_type(4), aligned(4)));
typedef float ff32x2u_t __attribute__((ext_vector_type(2), aligned(4)));

struct GemmF32Args {
    const float* x;
    const float* w;
    const void* bias;
    int bias_dtype;
    float* out;
    int M, N, K, KC, S;   // S chunks of KC (a multiple of 16; the last one may be short)
    int accumulate;
    int act;              // DKV_ACT_*, applied to the product plus bias
    int vec_out;          // rows of out are 16-byte aligned
};

__device__ __forceinline__ float gemm_bias(const GemmF32Args& a, int n) {
    return a.bias ? load_elem(a.bias, n, a.bias_dtype) : 0.0f;
}

// the activation kernels' arithmetic (model_ops.hip)
__device__ __forceinline__ float gemm_act(int act, float v) {
    if (act == DKV_ACT_GELU) {
        const float u = 0.7978845608028654f * (v + 0.044715f * v * v * v);
        return 0.5f * v * (1.0f + tanhf(u));
    }
    return act == DKV_ACT_RELU ? fmaxf(v, 0.0f) : v;
}

// outputs out[m][n .. n + 3] (+)= act(t + bias), up to column N - 1 of a row of N
__device__ __forceinline__ void gemm_store4(const GemmF32Args& a, int N, int m, int n, ff32x4_t t) {
    float* p = a.out + (int64_t)m * N + n;
    if (a.vec_out && n + 3 < N) {
        float4 v = make_float4(gemm_act(a.act, t[0] + gemm_bias(a, n)), gemm_act(a.act, t[1] + gemm_bias(a, n + 1)),
                               gemm_act(a.act, t[2] + gemm_bias(a, n + 2)), gemm_act(a.act, t[3] + gemm_bias(a, n + 3)));
        if (a.accumulate) {
            const float4 h = *reinterpret_cast<const float4*>(p);
            v = make_float4(h.x + v.x, h.y + v.y, h.z + v.z, h.w + v.w);
        }
        *reinterpret_cast<float4*>(p) = v;
        return;
    }
#pragma unroll
    for (int e = 0; e < 4; ++e)
        if (n + e < N) {
            const float v = gemm_act(a.act, t[e] + gemm_bias(a, n + e));
            p[e] = a.accumulate ? p[e] + v : v;
        }
}
// silu(g) * u, the SwiGLU kernel's arithmetic
__device__ __forceinline__ ff32x4_t gemm_glu(ff32x4_t g, ff32x4_t u) {
    ff32x4_t o;
#pragma unroll
    for (int e = 0; e < 4; ++e) o[e] = g[e] / (1.0f + __expf(-g[e])) * u[e];
    return o;
}

// A wave's tile: NW 16-column fragments of N by MB 16-row fragments of M.
// SPLIT: the workgroup's S waves take one chunk each of the same tile, and
// the sums meet in LDS; else its four waves own a 2 x 2 block of tiles (four
// tiles along N when MB * 16 covers M) and walk the chunks in order. Loads are
// vectors whatever K and the alignment (4-byte aligned 16-byte loads; element
// by element only where a group ends past K). GLU (layout 1): w
// holds N / 2 gate rows, then N / 2 up rows; the second half of the fragments
// are the up rows of the first half's, and out[M][N / 2] = silu(gate) * up.
template <int WL, int NW, int MB, bool SPLIT, bool GLU>
__global__ void __launch_bounds__(SPLIT ? 1024 : 256, SPLIT ? 4 : 2) gemm_f32_kernel(GemmF32Args a, int two_by_two) {
#pragma clang fp contract(off)
    static_assert(!GLU || (WL == 1 && NW % 2 == 0), "pairs of fragments of one layout");
    constexpr int FN = GLU ? NW / 2 : NW;   // fragments of the output
    constexpr int U = NW * MB >= 4 ? 2 : 4;                      // 16-k groups per register set
    extern __shared__ __align__(16) float red[];                 // SPLIT: [S][NW * MB][64 lanes][4]
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / WAVE), lane = threadIdx.x % WAVE;
    const int col = lane % 16, j = lane / 16;
    int tn = blockIdx.x, tm = blockIdx.y;
    if (!SPLIT) {
        tn = two_by_two ? 2 * tn + (wave & 1) : 4 * tn + wave;
        tm = two_by_two ? 2 * tm + (wave >> 1) : tm;
    }
    const int K = a.K, N = a.N, NO = GLU ? N / 2 : N;
    const int n0 = tn * 16 * FN, m0 = tm * 16 * MB;
    if (!SPLIT && (n0 >= NO || m0 >= a.M)) return;
    // rows past M and columns past N reread the last one; their products are never stored
    const float* xp[MB];
#pragma unroll
    for (int b = 0; b < MB; ++b) xp[b] = a.x + (int64_t)min(m0 + 16 * b + col, a.M - 1) * K;
    const float* wp[WL ? NW : 1];
    if constexpr (WL) {
#pragma unroll
        for (int f = 0; f < NW; ++f) wp[f] = a.w + (int64_t)(min(n0 + 16 * (f % FN) + col, NO - 1) + f / FN * NO) * K;
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
            if (full || kg + 4 <= K) {
#pragma unroll
                for (int b = 0; b < MB; ++b) {
                    const ff32x4u_t v = *reinterpret_cast<const ff32x4u_t*>(xp[b] + kg);
                    r.x[u][b][0] = v[0], r.x[u][b][1] = v[1], r.x[u][b][2] = v[2], r.x[u][b][3] = v[3];
                }
                if constexpr (WL) {
#pragma unroll
                    for (int f = 0; f < NW; ++f) {
                        const ff32x4u_t v = *reinterpret_cast<const ff32x4u_t*>(wp[f] + kg);
                        r.w[u][f][0] = v[0], r.w[u][f][1] = v[1], r.w[u][f][2] = v[2], r.w[u][f][3] = v[3];
                    }
                } else {
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        const float* p = wp[0] + (int64_t)(kg + e) * N;
                        if constexpr (NW == 2) {
                            const ff32x2u_t v = *reinterpret_cast<const ff32x2u_t*>(p);
                            r.w[u][0][e] = v[0], r.w[u][1][e] = v[1];
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
            if (k + 16 * u < kend) {
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
        // wave w sums and stores the output subtiles w, w + S, ...
        for (int i = wave; i < FN * MB; i += a.S) {
            const int f = i / MB, b = i % MB, m = m0 + 16 * b + col;
            auto sum = [&](int ff) {
                ff32x4_t t = *reinterpret_cast<const ff32x4_t*>(red + ((ff * MB + b) * WAVE + lane) * 4);
                for (int c = 1; c < a.S; ++c) {
                    const ff32x4_t v = *reinterpret_cast<const ff32x4_t*>(red + (((c * NW + ff) * MB + b) * WAVE + lane) * 4);
#pragma unroll
                    for (int e = 0; e < 4; ++e) t[e] = t[e] + v[e];
                }
                return t;
            };
            ff32x4_t t = sum(f);
            if constexpr (GLU) t = gemm_glu(t, sum(FN + f));
            if (m >= a.M) continue;
            if constexpr (WL == 1 || NW == 1) {
                gemm_store4(a, NO, m, n0 + 16 * f + 4 * j, t);
            } else {
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const int n = n0 + NW * (4 * j + e) + f;
                    if (n < N) {
                        const float v = gemm_act(a.act, t[e] + gemm_bias(a, n));
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
            if constexpr (GLU) {
#pragma unroll
                for (int f = 0; f < FN; ++f) gemm_store4(a, NO, m, n0 + 16 * f + 4 * j, gemm_glu(tot[f][b], tot[FN + f][b]));
            } else if constexpr (WL == 1 || NW == 1) {
#pragma unroll
                for (int f = 0; f < NW; ++f) gemm_store4(a, N, m, n0 + 16 * f + 4 * j, tot[f][b]);
            } else {   // the lane holds 4 NW consecutive columns: n0 + NW (4 j + e) + f
#pragma unroll
                for (int v = 0; v < NW; ++v) {
                    ff32x4_t t;
#pragma unroll
                    for (int e = 0; e < 4; ++e) t[e] = tot[(4 * v + e) % NW][b][(4 * v + e) / NW];
                    gemm_store4(a, N, m, n0 + 4 * NW * j + 4 * v, t);
                }
            }
        }
    }
}

// Many rows (K % 32 == 0): a workgroup of 2 x 2 waves, each with a tile of NW
// fragments of N by MB of M, shares its operands through LDS. Straight from
// L1 and L2 the waves' own loads (as above) run into the caches' bandwidth,
// about 5 TB/s: every 16 k of a 32 x 32 tile are 4 KB for 512 cycles of MFMA
// (the distilgpt2 head at 1000 rows 879 -> 769 us, its 2304 columns 81 -> 57).
// The 1 KB pieces come in by direct-to-LDS loads, three stages of one or two
// groups of 16 k in rotation, in the order of the operand reads: a 16-row
// fragment's lane (col, j) holds row col, k 4 j .. + 3; of a layout-0 w, piece
// e of 64 columns holds columns 4 col .. + 3 of row 4 j + e, and component f
// of a lane is its operand for the columns 4 i + f.
template <int WL, int NW, int MB, bool GLU>
__global__ void __launch_bounds__(256, 2) gemm_f32_lds_kernel(GemmF32Args a) {
#pragma clang fp contract(off)
    static_assert(!GLU || WL == 1, "SwiGLU weights are rows");
    constexpr int FN = GLU ? NW / 2 : NW;             // output fragments per wave
    constexpr int KS = NW == 4 ? 1 : 2, ST = 3;       // groups per stage, stages: 48 KB, so two workgroups per CU
    constexpr int WP = 2 * NW, XP = 2 * MB, PIECES = WP + XP;   // 1 KB pieces of a group
    constexpr int LPW = KS * PIECES / 4;              // loads per wave per stage
    extern __shared__ __align__(16) char lds[];       // [ST][KS][PIECES][1 KB]
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / WAVE), lane = threadIdx.x % WAVE;
    const int col = lane % 16, j = lane / 16, wn = wave & 1, wm = wave >> 1;
    const int K = a.K, N = a.N, NO = GLU ? N / 2 : N;
    const int n0 = blockIdx.x * 32 * FN, m0 = blockIdx.y * 32 * MB;   // the workgroup's tile
    // This wave's pieces: w pieces wave, wave + 4, ... and x pieces likewise. Rows past M and columns past N
    // reread the last one; their products are never stored.
    const char* base[PIECES / 4];
    uint32_t off[PIECES / 4];
    int64_t step[PIECES / 4];
#pragma unroll
    for (int x = 0; x < PIECES / 4; ++x) {
        const int p = 4 * x + wave;
        if (4 * x < WP && WL == 1) {          // fragment p: wave tile p / NW, its fragment p % NW
            const int f = p % NW, nf = n0 + 16 * (FN * (p / NW) + f % FN), up = f / FN;
            base[x] = reinterpret_cast<const char*>(a.w + ((int64_t)up * NO + min(nf, NO - 1)) * K);
            off[x] = (uint32_t)((min(nf + col, NO - 1) - min(nf, NO - 1)) * K + 4 * j) * 4;
            step[x] = 64;
        } else if (4 * x < WP) {              // 64 columns p / 4, row 4 j + p % 4
            const int nc = n0 + 64 * (p / 4);
            base[x] = reinterpret_cast<const char*>(a.w + (int64_t)(p % 4) * N + min(nc, N - 4));
            off[x] = (uint32_t)(4 * j * N + min(nc + 4 * col, N - 4) - min(nc, N - 4)) * 4;
            step[x] = 64 * (int64_t)N;
        } else {
            const int mf = m0 + 16 * (p - WP);
            base[x] = reinterpret_cast<const char*>(a.x + (int64_t)min(mf, a.M - 1) * K);
            off[x] = (uint32_t)((min(mf + col, a.M - 1) - min(mf, a.M - 1)) * K + 4 * j) * 4;
            step[x] = 64;
        }
    }
    const int NS = K / (16 * KS);
    auto issue = [&](int i) {
        const uint32_t to = lds_offset(lds + (i % ST) * (KS * PIECES * 1024));
#pragma unroll
        for (int g = 0; g < KS; ++g)
#pragma unroll
            for (int x = 0; x < PIECES / 4; ++x)
                dma_b128<false>(base[x] + (i * KS + g) * step[x], off[x], to + (g * PIECES + 4 * x + wave) * 1024);
    };
    ff32x4_t acc[NW][MB], tot[NW][MB];
    auto clear = [&]() {
#pragma unroll
        for (int f = 0; f < NW; ++f)
#pragma unroll
            for (int b = 0; b < MB; ++b) acc[f][b] = ff32x4_t{0.f, 0.f, 0.f, 0.f};
    };
    // A group's operands are read one group ahead of its products. When the group read next starts a stage:
    // that stage's loads are done once at most the later one's remain; every wave holds the operands of the
    // stage before (the wait covers its LDS reads), so after the barrier that stage's room takes new loads.
    struct Ops {
        ff32x4_t w[4], x[MB];   // layout 1: w[fragment]; layout 0: w[step]
    };
    auto read = [&](Ops& o, int g) {
        const char* s = lds + (g / KS % ST * KS + g % KS) * (PIECES * 1024) + lane * 16;
#pragma unroll
        for (int b = 0; b < MB; ++b) o.x[b] = *reinterpret_cast<const ff32x4_t*>(s + (WP + MB * wm + b) * 1024);
#pragma unroll
        for (int q = 0; q < (WL == 1 ? NW : 4); ++q)   // layout 0, NW == 2: the waves share the 64 columns' pieces
            o.w[q] = *reinterpret_cast<const ff32x4_t*>(s + ((WL == 1 || NW == 4 ? NW * wn : 0) + q) * 1024);
    };
    auto advance = [&](int st) {
        if (st + 1 < NS) wait_loads_barrier<LPW>();
        else wait_loads_barrier<0>();
        if (st + ST - 1 < NS) issue(st + ST - 1);
    };
    int left = a.KC / 16;   // groups until the chunk ends
    bool first = true;
    auto products = [&](const Ops& o, bool last) {
#pragma unroll
        for (int e = 0; e < 4; ++e)
#pragma unroll
            for (int f = 0; f < NW; ++f) {
                // layout 0: component f of the wave's 64 columns, or 2 wn + f of the shared ones
                const float w = WL == 1 ? o.w[f][e] : NW == 4 ? o.w[e][f] : wn ? o.w[e][2 + f % 2] : o.w[e][f % 2];
#pragma unroll
                for (int b = 0; b < MB; ++b)
                    acc[f][b] = __builtin_amdgcn_mfma_f32_16x16x4f32(w, o.x[b][e], acc[f][b], 0, 0, 0);
            }
        if (--left == 0 || last) {   // a chunk ends
            left = a.KC / 16;
#pragma unroll
            for (int f = 0; f < NW; ++f)
#pragma unroll
                for (int b = 0; b < MB; ++b) {
                    if (first) tot[f][b] = acc[f][b];
                    else
#pragma unroll
                        for (int e = 0; e < 4; ++e) tot[f][b][e] = tot[f][b][e] + acc[f][b][e];
                }
            first = false;
            clear();
        }
    };
    clear();
#pragma unroll
    for (int i = 0; i < ST; ++i)
        if (i < NS) issue(i);
    if (NS > 2) wait_loads_barrier<2 * LPW>();
    else if (NS == 2) wait_loads_barrier<LPW>();
    else wait_loads_barrier<0>();
    const int G = K / 16;
    Ops o0, o1;
    read(o0, 0);
    for (int g = 0; g < G; g += 2) {
        if (g + 1 < G) {
            if (KS == 1) advance(g + 1);
            read(o1, g + 1);
        }
        products(o0, g + 1 == G);
        if (g + 1 == G) break;
        if (g + 2 < G) {
            advance((g + 2) / KS);
            read(o0, g + 2);
        }
        products(o1, g + 2 == G);
    }
#pragma unroll
    for (int b = 0; b < MB; ++b) {
        const int m = m0 + 16 * (MB * wm + b) + col;
        if (m >= a.M) continue;
        if constexpr (WL == 1) {
#pragma unroll
            for (int f = 0; f < FN; ++f) {
                ff32x4_t t = tot[f][b];
                if constexpr (GLU) t = gemm_glu(t, tot[FN + f][b]);
                gemm_store4(a, NO, m, n0 + 16 * (FN * wn + f) + 4 * j, t);
            }
        } else if constexpr (NW == 4) {   // the lane holds 16 consecutive columns
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                const ff32x4_t t = {tot[0][b][v], tot[1][b][v], tot[2][b][v], tot[3][b][v]};
                gemm_store4(a, N, m, n0 + 64 * wn + 16 * j + 4 * v, t);
            }
        } else {                          // columns 4 (4 j + e) + 2 wn + f
#pragma unroll
            for (int e = 0; e < 4; ++e)
#pragma unroll
                for (int f = 0; f < NW; ++f) {
                    const int n = n0 + 4 * (4 * j + e) + 2 * wn + f;
                    if (n < N) {
                        const float v = gemm_act(a.act, tot[f][b][e] + gemm_bias(a, n));
                        float* p = a.out + (int64_t)m * N + n;
                        *p = a.accumulate ? *p + v : v;
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

template <int WL, int NW, int MB, bool SPLIT, bool GLU>
static int launch_f32(const GemmF32Args& a, bool two_by_two, hipStream_t st) {
    const int FN = GLU ? NW / 2 : NW, NO = GLU ? a.N / 2 : a.N;
    const int64_t tn = (NO + 16 * FN - 1) / (16 * FN), tm = (a.M + 16 * MB - 1) / (16 * MB);
    const int64_t gx = SPLIT ? tn : two_by_two ? (tn + 1) / 2 : (tn + 3) / 4;
    const int64_t gy = !SPLIT && two_by_two ? (tm + 1) / 2 : tm;
    const size_t lds = SPLIT ? sizeof(float) * 256 * (size_t)a.S * NW * MB : 0;
    auto kfn = gemm_f32_kernel<WL, NW, MB, SPLIT, GLU>;
    static size_t lds_done[16] = {};
    if (!reserve_lds(reinterpret_cast<const void*>(kfn), lds, lds_done))
        return fail(DKV_ELAUNCH, "dkv_gemm_f32: cannot reserve " + std::to_string(lds) + " B of LDS");
    hipLaunchKernelGGL(kfn, dim3((unsigned)gx, (unsigned)gy), dim3(SPLIT ? 64 * a.S : 256), lds, st, a, (int)two_by_two);
    return check_launch("dkv_gemm_f32");
}
template <int WL, int NW, int MB, bool GLU>
static int launch_split(const GemmF32Args& a, bool split, hipStream_t st) {
    return split ? launch_f32<WL, NW, MB, true, GLU>(a, false, st) : launch_f32<WL, NW, MB, false, GLU>(a, false, st);
}

template <int WL, int NW, bool GLU>
static int launch_lds(const GemmF32Args& a, hipStream_t st) {
    const int FN = GLU ? NW / 2 : NW, NO = GLU ? a.N / 2 : a.N;
    const size_t lds = 48 * 1024;   // three stages of two (NW = 2) or one (NW = 4) 16-k groups
    auto kfn = gemm_f32_lds_kernel<WL, NW, NW, GLU>;
    static size_t lds_done[16] = {};
    if (!reserve_lds(reinterpret_cast<const void*>(kfn), lds, lds_done))
        return fail(DKV_ELAUNCH, "dkv_gemm_f32: cannot reserve " + std::to_string(lds) + " B of LDS");
    hipLaunchKernelGGL(kfn, dim3((unsigned)((NO + 32 * FN - 1) / (32 * FN)), (unsigned)((a.M + 32 * NW - 1) / (32 * NW))),
                       dim3(256), lds, st, a);
    return check_launch("dkv_gemm_f32");
}

// Few rows: one fragment of w (or a gate and an up one) per wave, every row
// beside it, so w is read once. (A 3072 x 576 weight at a 4-byte aligned
// address, 1000 rows: 230 us with one output per thread, 495 with 16 x 16
// tiles and loads element by element, now 64.) From 65 rows on, through LDS where K and the
// alignment allow (`lds`): 64 x 64 per wave where that gives every SIMD a
// wave, else 32 x 32; without LDS 32 x 32 (16 x 64 where a layout-0 row has
// an odd number of columns), whose chunks go to the waves of a workgroup when
// the tiles leave half of the SIMDs without a wave.
template <int WL, bool GLU>
static int launch_f32_wl(const GemmF32Args& a, bool lds, hipStream_t st) {
    constexpr int F = GLU ? 2 : 1;
    const bool split = a.S > 1;
    // Single fragments also for more rows where larger tiles would leave SIMDs without a wave:
    // - up to 64 rows, when the (fragment, chunk) pairs are fewer than the 1024 SIMDs (33 / 64 rows of 768 x 768
    //   9.2 / 10.3 -> 4.6 / 4.7 us, of 768 x 3072 32 / 35 -> 11.4 / 11.7; 3072 x 768, 1152 pairs, 17 rows 6.0 / 6.6;
    //   4096 x 4096, 1024 pairs, 64 rows 36 / 81: w is read once per 16 rows);
    // - one chain of at most 8 groups (K < 128), up to 2048 fragments: a tile's time is its MFMAs' (64 / 256 x 64 for
    //   1000 rows 5.3 / 5.4 us through LDS -> 3.2 / 3.4; 1000 x 112 for 512 rows (2016 fragments) 6.8 -> 5.3, for
    //   1000 (3969) 7.2 / 8.6).
    const int64_t frags = (a.N + 15) / 16;
    const bool small = (a.M <= 64 && frags * a.S < 1024) || (a.K < 128 && frags * ((a.M + 15) / 16) <= 2048);
    if (a.M <= 16 || small) return launch_split<WL, F, 1, GLU>(a, split, st);
    if (a.M <= 32) return launch_split<WL, F, 2, GLU>(a, split, st);
    if constexpr (!GLU)   // (a pair's partials of 64 rows would take more LDS than two workgroups' share)
        if (a.M <= 64) return launch_split<WL, F, 4, GLU>(a, split, st);
    const int64_t w44 = (int64_t)((a.N + 63) / 64) * ((a.M + 63) / 64), w22 = (int64_t)((a.N + 31) / 32) * ((a.M + 31) / 32);
    const bool walk = w22 >= 512 || !split;
    if (lds && walk) return w44 >= 1024 ? launch_lds<WL, 4, GLU>(a, st) : launch_lds<WL, 2, GLU>(a, st);
    if constexpr (WL == 0)
        if (a.N % 2) return walk ? launch_f32<WL, 1, 4, false, false>(a, false, st) : launch_split<WL, 1, 4, false>(a, true, st);
    return walk ? launch_f32<WL, 2, 2, false, GLU>(a, true, st) : launch_f32<WL, 2, 2, true, GLU>(a, false, st);
}

static int gemm_f32(const float* x, const float* w, int32_t w_layout, int32_t M, int32_t N, int32_t K, const void* bias,
                    int32_t bias_dtype, int32_t act, float* out, int32_t accumulate, dkv_stream_t stream) {
    const ChunksF32 c = gemm_f32_chunks(N, K);
    auto aligned = [](const void* p) { return reinterpret_cast<uintptr_t>(p) % 16 == 0; };
    GemmF32Args a;
    a.x = x, a.w = w, a.bias = bias, a.bias_dtype = bias_dtype, a.out = out;
    a.M = M, a.N = N, a.K = K, a.KC = c.KC, a.S = c.S, a.accumulate = accumulate, a.act = act;
    const bool glu = act == DKV_ACT_SWIGLU;
    a.vec_out = (glu ? N / 2 : N) % 4 == 0 && aligned(out);
    const bool lds = K % 32 == 0 && aligned(x) && aligned(w) && (w_layout == 1 || N % 4 == 0);
    hipStream_t st = as_stream(stream);
    if (glu) return launch_f32_wl<1, true>(a, lds, st);
    return w_layout == 1 ? launch_f32_wl<1, false>(a, lds, st) : launch_f32_wl<0, false>(a, lds, st);
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
    return gemm_f32(x, w, w_layout, M, N, K, bias, bias_dtype, DKV_ACT_NONE, out, accumulate, stream);
}

extern "C" int32_t dkv_gemm_f32_act_ok(const float* x, const float* w, int32_t w_layout, int32_t N, int32_t K,
                                       int32_t act) {
    if (act != DKV_ACT_SWIGLU) return act == DKV_ACT_GELU || act == DKV_ACT_RELU;
    auto aligned = [](const void* p) { return reinterpret_cast<uintptr_t>(p) % 16 == 0; };
    return w_layout == 1 && N % 2 == 0 && K % 4 == 0 && aligned(x) && aligned(w);
}

extern "C" int dkv_gemm_f32_act(const float* x, const float* w, int32_t w_layout, int32_t M, int32_t N, int32_t K,
                                const void* bias, int32_t bias_dtype, int32_t act, float* out, dkv_stream_t stream) {
    DKV_REQUIRE(x && w && out && N > 0 && K > 0 && (w_layout == 0 || w_layout == 1), "dkv_gemm_f32_act: bad arguments");
    DKV_REQUIRE(!bias || bias_dtype == DKV_F32 || bias_dtype == DKV_BF16, "dkv_gemm_f32_act: bad bias dtype");
    DKV_REQUIRE(M <= 65535 * 16, "dkv_gemm_f32_act: too many rows for one launch");
    DKV_REQUIRE(dkv_gemm_f32_act_ok(x, w, w_layout, N, K, act) && !(act == DKV_ACT_SWIGLU && bias),
                "dkv_gemm_f32_act: SwiGLU needs w[N][K], even N, K % 4 == 0, 16-byte aligned operands and no bias");
    if (M <= 0) return DKV_OK;
    return gemm_f32(x, w, w_layout, M, N, K, bias, bias_dtype, act, out, 0, stream);
}

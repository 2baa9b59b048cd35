// Paged full-cache append and causal attention over it.
// Reference: draftkv/paged.py:76-176 (cache), draftkv/llama.py:202-218 and
// gpt2.py/model.py equivalents (read + masked softmax attention).
#include <algorithm>

#include "dkv_common.h"
#include "paged_attn.h"

namespace dkv {

// ---------------------------------------------------------------- append
__global__ void __launch_bounds__(256) paged_append_kernel(dkv_paged_t c, int layer, const void* __restrict__ k,
                                                           const void* __restrict__ v, int in_dtype, int T,
                                                           const int32_t* __restrict__ start,
                                                           const int32_t* __restrict__ count) {
    const int t = blockIdx.x, s = blockIdx.y;
    if (count && t >= count[s]) return;
    const int pos = start[s] + t;
    const int32_t blk = paged_block(c, s, layer, pos);
    const int off = pos % c.block_size;
    const int HD = c.n_kv_heads * c.head_dim;
    const int64_t src = ((int64_t)s * T + t) * HD;
    for (int i = threadIdx.x; i < HD; i += blockDim.x) {
        const int h = i / c.head_dim, d = i % c.head_dim;
        const float kv = load_elem(k, src + i, in_dtype);
        const float vv = load_elem(v, src + i, in_dtype);
        const int64_t ko = paged_k_off(c, blk, off, h, d), vo = paged_v_off(c, blk, off, h, d);
        if (c.dtype == DKV_BF16) {
            static_cast<uint16_t*>(c.pool)[ko] = f32_to_bf16_rne(kv);
            static_cast<uint16_t*>(c.pool)[vo] = f32_to_bf16_rne(vv);
        } else {
            static_cast<float*>(c.pool)[ko] = kv;
            static_cast<float*>(c.pool)[vo] = vv;
        }
    }
}

__device__ __forceinline__ float load_x(const float* p, int64_t i) { return p[i]; }
__device__ __forceinline__ float load_x(const uint16_t* p, int64_t i) { return bf16_to_f32(p[i]); }

// The same for prompts into 16-token blocks: a workgroup owns one block of
// one (sequence, KV head). Row by row the transposed V takes one 2- or 4-byte
// store per element, 32 or 64 bytes apart; here a thread holds a channel's 16
// tokens and stores their whole run (float32 rows, 4000 tokens: 8 heads of 128
// in bf16 23.1 -> 11.2 us, 12 of 64 in float32 29.1 -> 12.8). Its chain of
// loads and stores is the longer one, 4.0 to 4.7 us for the smallest prompts
// against 2.8: it is for T >= 64 and as many elements as where the two meet,
// 200k in a float32 cache, in a bf16 one 256k of bf16 rows or 600k of float32
// rows (1000 tokens of 3 heads of 64: 4.4 / 4.2, 3.9 / 4.2 and 3.5 / 4.5; 3200
// of them 8.1 / 5.6, 6.7 / 4.7 and 6.1 / 5.1). Tokens of the block outside
// this append keep what they hold.
template <bool BF16, class X>
__global__ void __launch_bounds__(128) paged_append_block_kernel(dkv_paged_t c, int layer, const X* __restrict__ k,
                                                                 const X* __restrict__ v, int T,
                                                                 const int32_t* __restrict__ start,
                                                                 const int32_t* __restrict__ count) {
    const int h = blockIdx.y, s = blockIdx.z, D = c.head_dim;
    const int s0 = start[s], n = min(count ? count[s] : T, T);
    const int b = s0 / 16 + blockIdx.x;                       // block of the sequence
    const int p0 = max(16 * b, s0), p1 = min(16 * b + 16, s0 + n);   // the positions it takes
    if (p0 >= p1) return;
    const int32_t blk = paged_block(c, s, layer, 16 * b);
    const int64_t src = (((int64_t)s * T + (16 * b - s0)) * c.n_kv_heads + h) * D, row = (int64_t)c.n_kv_heads * D;
    const int o0 = p0 - 16 * b, o1 = p1 - 16 * b;
    for (int d = threadIdx.x; d < D; d += blockDim.x) {
        // every load before the first store, none of them behind a branch: tokens outside reread the nearest one
        float xk[16], xv[16];
#pragma unroll
        for (int o = 0; o < 16; ++o) {
            const int64_t at = src + min(max(o, o0), o1 - 1) * row + d;
            xk[o] = load_x(k, at);
            xv[o] = load_x(v, at);
        }
#pragma unroll
        for (int o = 0; o < 16; ++o)
            if (o >= o0 && o < o1) {
                const int64_t at = paged_k_off(c, blk, o, h, d);
                if constexpr (BF16) static_cast<uint16_t*>(c.pool)[at] = f32_to_bf16_rne(xk[o]);
                else static_cast<float*>(c.pool)[at] = xk[o];
            }
        const int64_t at = paged_v_off(c, blk, 0, h, d);
        if (o0 == 0 && o1 == 16) {
            if constexpr (BF16) {
                uint32_t w[8];
#pragma unroll
                for (int o = 0; o < 8; ++o)
                    w[o] = (uint32_t)f32_to_bf16_rne(xv[2 * o]) | (uint32_t)f32_to_bf16_rne(xv[2 * o + 1]) << 16;
                uint4* p = reinterpret_cast<uint4*>(static_cast<uint16_t*>(c.pool) + at);
                p[0] = make_uint4(w[0], w[1], w[2], w[3]);
                p[1] = make_uint4(w[4], w[5], w[6], w[7]);
            } else {
                float4* p = reinterpret_cast<float4*>(static_cast<float*>(c.pool) + at);
#pragma unroll
                for (int o = 0; o < 4; ++o) p[o] = make_float4(xv[4 * o], xv[4 * o + 1], xv[4 * o + 2], xv[4 * o + 3]);
            }
        } else {
#pragma unroll
            for (int o = 0; o < 16; ++o)
                if (o >= o0 && o < o1) {
                    if constexpr (BF16) static_cast<uint16_t*>(c.pool)[at + o] = f32_to_bf16_rne(xv[o]);
                    else static_cast<float*>(c.pool)[at + o] = xv[o];
                }
        }
    }
}

// ---------------------------------------------------------------- attention
// Grid: x = chunk * n_qtiles + qtile, y = kv head, z = sequence.
// A block owns QB query rows (query row r -> step t = r / G, head h*G + r%G)
// and the keys [chunk*CH, min((chunk+1)*CH, len)). Keys are walked in tiles
// of KT at fixed absolute offsets; per query row the arithmetic (dot order,
// tile max/sum order, rescale sequence) depends only on absolute key indices,
// never on T or on how many rows share the block, so a row's partial is
// bit-identical whether it is computed in a verify pass (T = gamma+1) or in a
// one-token decode step. Masked keys contribute exact zeros. The cache ends
// at start + count (count null: all T rows were appended); positions past it
// are never read as keys -- their pages may hold stale bytes, and 0 * NaN is
// NaN -- and a padding row (t >= count) attends over the whole cache.
constexpr int QB = 16;
constexpr int KT = 32;
constexpr int MAXD = 128;   // LDS tiles stay under 64 KB

__global__ void __launch_bounds__(256) paged_attn_kernel(dkv_paged_t c, int layer, const float* __restrict__ q,
                                                         int T, int Hq, const int32_t* __restrict__ start,
                                                         const int32_t* __restrict__ count, int CH, int n_chunks,
                                                         int n_qtiles, float scale, float* __restrict__ part) {
    const int chunk = blockIdx.x / n_qtiles, qtile = blockIdx.x % n_qtiles;
    const int h = blockIdx.y, s = blockIdx.z;
    const int D = c.head_dim, G = Hq / c.n_kv_heads;
    const int s0 = start[s];
    const int len = s0 + (count ? count[s] : T);  // cache holds positions 0..len-1
    const int k_begin = chunk * CH;
    if (k_begin >= len) return;
    const int k_end = min(k_begin + CH, len);
    const int n_rows = T * G;
    const int r0 = qtile * QB;
    if (r0 >= n_rows) return;
    const int nr = min(QB, n_rows - r0);
    // last key any of this block's rows may see
    const int max_qpos = s0 + (r0 + nr - 1) / G;
    if (k_begin > max_qpos) return;

    extern __shared__ float smem[];
    float* sQ = smem;                               // [QB][D]
    float* sK = sQ + QB * D;                        // [KT][D+1]
    float* sV = sK + KT * (D + 1);                  // [KT][D]
    float* sS = sV + KT * D;                        // [QB][KT]
    float* sM = sS + QB * KT;                       // [QB] running max
    float* sL = sM + QB;                            // [QB] running sum
    float* sA = sL + QB;                            // [QB] rescale factor of this tile

    const int tid = threadIdx.x;
    for (int i = tid; i < QB * D; i += blockDim.x) {
        const int r = i / D, d = i % D;
        float val = 0.0f;
        if (r < nr) {
            const int rr = r0 + r, t = rr / G, hq = h * G + rr % G;
            val = q[(((int64_t)s * T + t) * Hq + hq) * D + d];
        }
        sQ[i] = val;
    }
    if (tid < QB) {
        sM[tid] = -INFINITY;
        sL[tid] = 0.0f;
    }
    // accumulators: outputs o = tid + 256*j (row o / D, dim o % D)
    constexpr int MAXACC = QB * MAXD / 256;
    float acc[MAXACC];
#pragma unroll
    for (int j = 0; j < MAXACC; ++j) acc[j] = 0.0f;
    const int n_out = QB * D;

    const int kend_eff = min(k_end, max_qpos + 1);
    for (int kt = k_begin; kt < kend_eff; kt += KT) {
        __syncthreads();
        // load K and V tiles (keys kt .. kt+KT-1, zero past the cache)
        for (int i = tid; i < KT * D; i += blockDim.x) {
            const int j = i / D, d = i % D;
            const int pos = kt + j;
            float kv = 0.0f, vv = 0.0f;
            if (pos < len) {
                const int32_t blk = paged_block(c, s, layer, pos);
                const int off = pos % c.block_size;
                kv = load_elem(c.pool, paged_k_off(c, blk, off, h, d), c.dtype);
                vv = load_elem(c.pool, paged_v_off(c, blk, off, h, d), c.dtype);
            }
            sK[j * (D + 1) + d] = kv;
            sV[j * D + d] = vv;
        }
        __syncthreads();
        // scores
        for (int i = tid; i < QB * KT; i += blockDim.x) {
            const int r = i / KT, j = i % KT;
            const int pos = kt + j;
            float sc = -INFINITY;
            if (r < nr) {
                const int qpos = s0 + (r0 + r) / G;
                if (pos <= qpos && pos < len) {
                    float dot = 0.0f;
                    for (int d = 0; d < D; ++d) dot = fmaf(sQ[r * D + d], sK[j * (D + 1) + d], dot);
                    sc = dot * scale;
                }
            }
            sS[i] = sc;
        }
        __syncthreads();
        // online softmax per row: 16 lanes per row, fixed reduction tree
        {
            const int r = tid / 16, l16 = tid % 16;   // 256 threads = QB rows x 16
            float mx = -INFINITY;
            for (int j = l16; j < KT; j += 16) mx = fmaxf(mx, sS[r * KT + j]);
            for (int o = 8; o > 0; o >>= 1) mx = fmaxf(mx, __shfl_xor(mx, o, 16));
            const float m_old = sM[r];
            const float m_new = fmaxf(m_old, mx);
            float sum = 0.0f;
            for (int j = l16; j < KT; j += 16) {
                const float sc = sS[r * KT + j];
                const float p = (sc == -INFINITY) ? 0.0f : __expf(sc - m_new);
                sS[r * KT + j] = p;
                sum += p;
            }
            for (int o = 8; o > 0; o >>= 1) sum += __shfl_xor(sum, o, 16);
            __syncthreads();
            if (l16 == 0) {
                const float a = (m_old == -INFINITY) ? 0.0f : __expf(m_old - m_new);
                sA[r] = a;
                sL[r] = sL[r] * a + sum;
                sM[r] = m_new;
            }
        }
        __syncthreads();
        // PV
#pragma unroll
        for (int jj = 0; jj < MAXACC; ++jj) {
            const int o = tid + 256 * jj;
            if (o < n_out) {
                const int r = o / D, d = o % D;
                float a = acc[jj] * sA[r];
                for (int j = 0; j < KT; ++j) a = fmaf(sS[r * KT + j], sV[j * D + d], a);
                acc[jj] = a;
            }
        }
    }
    __syncthreads();
    // write partials: [((s*T + t)*Hq + hq) * n_chunks + chunk] * (D + 2)
#pragma unroll
    for (int jj = 0; jj < MAXACC; ++jj) {
        const int o = tid + 256 * jj;
        if (o < n_out) {
            const int r = o / D, d = o % D;
            if (r < nr) {
                const int rr = r0 + r, t = rr / G, hq = h * G + rr % G;
                float* p = part + ((((int64_t)s * T + t) * Hq + hq) * n_chunks + chunk) * (D + 2);
                p[d] = acc[jj];
                if (d == 0) {
                    p[D] = sM[r];
                    p[D + 1] = sL[r];
                }
            }
        }
    }
}

// ---------------------------------------------------------------- MFMA path
// bf16 cache with 16-token blocks, D = 64 or 128. A workgroup owns one
// (sequence, KV head, key range) and W q-tiles of 16 query rows, one wave per
// q-tile, and walks the range 32 keys (two blocks) per step:
//   S^T[16 keys][16 rows] = K[16 keys][D] . Q^T     (v_mfma_f32_16x16x32_bf16)
//   O^T[16 d][16 rows]   += V^T[16 d][32 keys] . P^T
// Q and P are split into bf16 hi + lo parts (two MFMAs each), which keeps the
// products at ~16 mantissa bits against the exact bf16 K/V. In the S^T
// accumulator a lane holds keys 4*(l/16)+r of one query row l%16; the PV
// B operand wants 8 keys of one row per lane, so the k-slots of the PV
// product are ordered {4j..4j+3, 16+4j..16+4j+3} (j = l/16) and the
// probabilities never leave their lane. In k-step st of the QK product lane
// group j holds d in [32 st + 8 j, +8), so a step's K load reads 64
// contiguous bytes of each key row.
//
// Staging. The K and V of a step go to LDS through direct-to-LDS loads
// (global_load_lds_dwordx4), S steps deep, so HBM latency hides behind the
// products of earlier steps without holding registers, and the workgroup
// reads each byte of its range from HBM once whatever the number of q-tiles.
// K lands in the order of the QK A operand (slot (tile, k-step)
// = 1 KB, 16 B per lane), so an operand read is one conflict-free
// ds_read_b128; V^T keeps its layout but for a swap (v_half). The loads are
// issued from inline asm and waited for by hand (s_waitcnt vmcnt + s_barrier):
// the compiler's own tracking of LDS DMA would make every LDS read wait for
// all loads in flight, prefetches included.
//
// Arithmetic: units of up to 128 keys (paged_attn.h), four 32-key steps with
// an online softmax inside the unit. Floating-point contraction is off, so
// every instantiation rounds alike.
//
// Launch shapes. Decode and verify stream K and V once: one q-tile per wave,
// as many waves as q-tiles (up to 8), two stages (32 KB beside the block ids:
// four workgroups per CU hide the latency), non-temporal loads; where the (rows, chunk) pairs do
// not fill the chip every unit is a workgroup of its own, its four steps in
// flight at once. Prompts (more than 8 q-tiles per KV head) are bound by the
// softmax's VALU work, the LDS reads and the matrix cores together, so what
// counts is waves in flight: 168 registers for three per SIMD, uniform
// branches around masking and rescaling, loads that are cached (each K/V
// byte is read by many workgroups) and kept to one XCD's L2 per (sequence, KV
// head) pair where the pairs are a multiple of 8. Two q-tiles per wave, which
// halve the LDS reads, measured slower (256 registers: 486 against 393 us).
typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef float f32x4_t __attribute__((ext_vector_type(4)));
typedef float f32x4u_t __attribute__((ext_vector_type(4), aligned(4)));   // callers' pointers need 4-byte alignment only

typedef __bf16 bf16x2_t __attribute__((ext_vector_type(2)));
typedef float f32x2_t __attribute__((ext_vector_type(2)));
// (a, b) into elements k, k + 1 of the bf16 high and low parts, each rounded
// to nearest even (v_cvt_pk_bf16_f32)
__device__ __forceinline__ void split_pair(float a, float b, bf16x8_t& hi, bf16x8_t& lo, int k) {
    const bf16x2_t h = __builtin_convertvector((f32x2_t){a, b}, bf16x2_t);
    const uint32_t u = __builtin_bit_cast(uint32_t, h);
    const bf16x2_t l = __builtin_convertvector(
        (f32x2_t){a - __uint_as_float(u << 16), b - __uint_as_float(u & 0xffff0000u)}, bf16x2_t);
    hi[k] = h[0], hi[k + 1] = h[1], lo[k] = l[0], lo[k + 1] = l[1];
}

template <int D>
struct VerifyStage {
    static constexpr int NSTEP = D / 32;               // k-steps of the QK product
    static constexpr int K_BYTES = 2 * NSTEP * 1024;   // two 16-key tiles, operand order
    static constexpr int V_BLOCK = D * 16 * 2;         // one block's V^T of one head
    static constexpr int NVI = V_BLOCK / 1024;         // 1 KB loads per V block
    static constexpr int NI = 2 * NSTEP + 2 * NVI;     // 1 KB loads per step
    static constexpr int BYTES = K_BYTES + 2 * V_BLOCK;
};

// Staged V^T: 32 bytes per row, keys 0-7 and 8-15 of the block, swapped in
// rows 4-7 of every 8. A PV operand read takes one half of 16 rows at a time;
// in plain order those lie 32 bytes apart, on half of the LDS banks (a quarter
// of a prompt's time). Conflict cycles per LDS instruction: nine rows 8.5 ->
// 3.3, a prompt now 3.6.
__device__ __forceinline__ int v_half(int row, int half) { return half ^ (row >> 2 & 1); }

// The lane's index, worked out where it is called: a value that is used at a
// walk's ends and in its rare branches only must not hold a register, or be
// spilled, along the walk.
__device__ __forceinline__ int lane_again() {
    int lane = __builtin_amdgcn_mbcnt_hi(~0u, __builtin_amdgcn_mbcnt_lo(~0u, 0u));
    asm volatile("" : "+v"(lane));
    return lane;
}

// The staged V^T of a step whose first `live` keys are the cache's last: the
// keys past them become zero (their probability is 0, and 0 * whatever the
// page holds could be NaN). 16-byte piece p: block, row, half.
template <int D>
__device__ __forceinline__ void zero_past(char* v, int live, int thread, int threads) {
    for (int p = thread; p < 4 * D; p += threads) {
        const int n = live - (16 * (p / (2 * D)) + 8 * v_half(p / 2, p & 1));   // live keys of the piece
        if (n >= 8) continue;
        uint16_t* e = reinterpret_cast<uint16_t*>(v + 16 * p);
        for (int k = max(n, 0); k < 8; ++k) e[k] = 0;
    }
}

// Running sums of a walking wave that stay in LDS: d-tiles of them (1 KB per
// wave), and with them the (m, l) of its 16 rows. The walk with D = 128 and
// four or eight waves needs a few registers more than the 128 that four waves
// per SIMD leave. Spilled to scratch, their reloads at each unit's end waited
// for every load in flight, the next step's K and V among them (Llama-3-8B
// heads, batch 32, T = 9 / 17: ctx 8k 199 / 338 -> 187 / 271 us, ctx 32k 710 /
// 1137 -> 680 / 976; 156 registers and three waves per SIMD instead: 211 / 358
// and 792 / 1311).
constexpr int fold_tiles(int D, int W, bool walk, bool nt) { return walk && nt && D == 128 ? W == 4 ? 1 : W == 8 ? 4 : 0 : 0; }
constexpr int fold_bytes(int tiles, int W) { return tiles ? W * (1024 * tiles + 16 * 8) : 0; }

template <int D, int W, int S, bool WALK, bool NT>
__global__ void __launch_bounds__(64 * W, W >= 4 && NT ? 4 : 3) paged_attn_mfma_kernel(PagedAttnArgs A) {
#pragma clang fp contract(off)
    using St = VerifyStage<D>;
    constexpr int NSTEP = St::NSTEP;
    constexpr int NDT = D / 16;        // d-tiles of the PV product
    constexpr int LPW = St::NI / W;    // loads per wave per step
    constexpr int TL = fold_tiles(D, W, WALK, NT), TR = WALK ? NDT - TL : 1;   // d-tiles of tot in LDS, in registers
    static_assert(St::NI % W == 0, "a step's loads split evenly over the waves");
    const dkv_paged_t& c = A.c;
    // wave index through readfirstlane: the q-tiles and everything derived
    // from them are then wave-uniform (scalar registers and branches)
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / WAVE), lane = threadIdx.x % WAVE;
    // grid (head x sequence, q-group, slot): the slot is the slowest index, so
    // the workgroups of the full slots are dispatched first and the short
    // last one fills the tail instead of splitting a round; of a prompt's
    // q-groups the last ones see the most keys and go first
    const int h = blockIdx.x % c.n_kv_heads, s = blockIdx.x / c.n_kv_heads;
    const int qg = A.group0 + gridDim.y - 1 - blockIdx.y, slot0 = blockIdx.z * A.run;
    const int T = A.T, Hq = A.Hq, G = __builtin_amdgcn_readfirstlane(Hq / c.n_kv_heads);
    const int s0 = __builtin_amdgcn_readfirstlane(A.start[s]);
    const int len = s0 + (A.count ? __builtin_amdgcn_readfirstlane(A.count[s]) : T);
    const int k_begin = slot0 * A.span;
    const int n_rows = T * G;
    const int col = lane % 16, jj = lane / 16;
    const int r0 = (qg * W + wave) * 16;   // the wave's first row
    const bool active = r0 < n_rows;       // wave-uniform
    const int r = r0 + col;
    const bool rvalid = r < n_rows;
    const int t = rvalid ? r / G : 0;
    const int64_t orow = ((int64_t)s * T + t) * Hq + h * G + (rvalid ? r % G : 0);
    // the group's last row bounds the keys any of its rows may see
    const int max_qpos = __builtin_amdgcn_readfirstlane(s0 + (min((qg + 1) * W * 16, n_rows) - 1) / G);
    if (k_begin >= len || k_begin > max_qpos) {   // uniform over the workgroup
        if (slot0 == 0 && len <= 0) {              // an empty cache: nothing to attend to
            const int ln = TL > 0 ? lane_again() : lane, row = r0 + ln % 16;
            if (row < n_rows)
                for (int d = ln / 16; d < D; d += 4)
                    A.out[(((int64_t)s * T + row / G) * Hq + h * G + row % G) * D + d] = 0.0f;
        }
        return;
    }
    // (the last workgroup's run may hold fewer slots)
    const int k_end = min(min(min(slot0 + A.run, A.n_slots) * A.span, len), max_qpos + 1);
    const int nsteps = (k_end - k_begin + 31) / 32;
    // this wave's rows: the last key any sees, and the last key all see
    const int wave_last = __builtin_amdgcn_readfirstlane(s0 + (min(r0 + 16, n_rows) - 1) / G);
    const int wave_all = __builtin_amdgcn_readfirstlane(min(s0 + r0 / G, len - 1));

    extern __shared__ __align__(16) char lds[];
    // block ids of the keys [k_begin, min(k_begin + 32 * nsteps, len))
    int32_t* sblk = reinterpret_cast<int32_t*>(lds + S * St::BYTES + fold_bytes(TL, W));
    // the wave's own: tile i of a lane at stot()[64 i], (m, l) of its row
    auto stot = [&](int lane) { return reinterpret_cast<f32x4_t*>(lds + S * St::BYTES) + wave * TL * WAVE + lane; };
    auto sml = [&](int lane) {
        return reinterpret_cast<float2*>(lds + S * St::BYTES + W * TL * 1024) + wave * 16 + lane % 16;
    };
    {
        const int32_t* btab = c.block_table + ((int64_t)s * c.n_layers + A.layer) * c.max_blocks + k_begin / 16;
        const int nblk = (min(k_begin + 32 * nsteps, len) - k_begin + 15) / 16;
        for (int i = threadIdx.x; i < nblk; i += 64 * W) sblk[i] = btab[i];
    }

    bf16x8_t qhi[NSTEP], qlo[NSTEP];
    {   // (rows past the last read row 0's query; nothing of theirs is stored). Loaded whole before any is used.
        const float* qr = A.q + orow * D + 8 * jj;
        f32x4_t v[NSTEP][2];
#pragma unroll
        for (int st = 0; st < NSTEP; ++st)
#pragma unroll
            for (int x = 0; x < 2; ++x) v[st][x] = *reinterpret_cast<const f32x4u_t*>(qr + 32 * st + 4 * x);
#pragma unroll
        for (int st = 0; st < NSTEP; ++st)
#pragma unroll
            for (int e = 0; e < 8; e += 2)   // scores come out scaled
                split_pair(v[st][e / 4][e % 4] * A.qscale, v[st][e / 4][e % 4 + 1] * A.qscale, qhi[st], qlo[st], e);
    }
    __syncthreads();   // block ids visible (no staging load is in flight yet)

    const char* pool = static_cast<const char*>(c.pool);
    const int64_t bel = 2 * paged_block_elems(c), kbase = (int64_t)h * 32 * D;   // bytes
    const int64_t vbase = ((int64_t)c.n_kv_heads + h) * 32 * D;
    // The lane's 16 bytes of a 1 KB load: of 16 K rows, 64 bytes each (row
    // col, chunk jj); of 32 V^T rows, row lane / 2, the two key halves of rows
    // 4 .. 7 of every 8 swapped
    const uint32_t klane = (uint32_t)(col * D + 8 * jj) * 2;
    const uint32_t vlane = (uint32_t)(lane / 2 * 16 + 8 * v_half(lane / 2, lane & 1)) * 2;
    // this wave's loads of a step: byte offset in the block, and which of the step's two blocks
    int64_t off[LPW];
    bool second[LPW];
#pragma unroll
    for (int x = 0; x < LPW; ++x) {
        const int i = wave * LPW + x, v = i - 2 * NSTEP;
        second[x] = i < 2 * NSTEP ? i >= NSTEP : v >= St::NVI;
        off[x] = i < 2 * NSTEP ? kbase + 64 * (i % NSTEP) : vbase + 1024 * (v % St::NVI);
    }
    // the loads of step j, into stage j % S
    auto issue = [&](int j) {
        const int kb = k_begin + 32 * j;
        const int32_t b0 = __builtin_amdgcn_readfirstlane(sblk[2 * j]);
        const int32_t b1 = (kb + 16 < len) ? __builtin_amdgcn_readfirstlane(sblk[2 * j + 1]) : b0;
        const char* g0 = pool + b0 * bel;
        const char* g1 = pool + b1 * bel;
        const uint32_t base = lds_offset(lds + (j % S) * St::BYTES);
#pragma unroll
        for (int x = 0; x < LPW; ++x) {
            const int i = wave * LPW + x;   // K tile a, k-step st, then V^T of block a, 1 KB piece pc
            dma_b128<NT>((second[x] ? g1 : g0) + off[x], i < 2 * NSTEP ? klane : vlane, base + i * 1024);
        }
    };

    f32x4_t acc[NDT], tot[TR];   // the current unit's sums, and the units before it
    float m_run, l_run, m_tot = -INFINITY, l_tot = 0.0f;
    auto clear = [&]() {
        m_run = -INFINITY;
        l_run = 0.0f;
#pragma unroll
        for (int i = 0; i < NDT; ++i) acc[i] = f32x4_t{0.f, 0.f, 0.f, 0.f};
    };
    // a slot's state out (lane: channels 16 dt + 4 jj .. + 3)
    auto store = [&](int slot, float m, float l, const f32x4_t* o) {
        const int ln = TL > 0 ? lane_again() : lane, jj = ln / 16, r = r0 + ln % 16;
        if (r >= n_rows) return;
        const int t = r / G;
        const int64_t orow = ((int64_t)s * T + t) * Hq + h * G + r % G;
        if (last_key(s0, t, len) >= A.span && A.n_slots > 1) {
            const int64_t ps = orow * A.n_slots + slot;
#pragma unroll
            for (int dt = 0; dt < NDT; ++dt) *reinterpret_cast<f32x4u_t*>(A.part + ps * D + 16 * dt + 4 * jj) = o[dt];
            if (jj == 0) A.ml[ps] = make_float2(m, l);
        } else if (slot == 0) {   // the row sees no other slot
#pragma unroll
            for (int dt = 0; dt < NDT; ++dt)
                *reinterpret_cast<f32x4u_t*>(A.out + orow * D + 16 * dt + 4 * jj) =
                    f32x4u_t{o[dt][0] / l, o[dt][1] / l, o[dt][2] / l, o[dt][3] / l};
        }
    };
    int slot = slot0;
    // a unit's end (l_run holds the lane's own keys: the four lane groups' sums meet here)
    auto unit_end = [&]() {
        if constexpr (!WALK) {
            store(slot++, m_run, lanegroup_sum(l_run), acc);
        } else {
            float fa, fb;
            const int lane = TL > 0 ? lane_again() : 0;
            if constexpr (TL > 0) m_tot = sml(lane)->x, l_tot = sml(lane)->y;
            m_tot = fold_max(m_tot, m_run, fa, fb);
            l_tot = fold_sum(l_tot, fa, lanegroup_sum(l_run), fb);
            if constexpr (TL > 0) *sml(lane) = make_float2(m_tot, l_tot);   // the four lane groups hold the same bits
#pragma unroll
            for (int i = 0; i < TR; ++i)
#pragma unroll
                for (int e = 0; e < 4; ++e) tot[i][e] = fold_sum(tot[i][e], fa, acc[i][e], fb);
#pragma unroll
            for (int i = 0; i < TL; ++i) {
                f32x4_t x = stot(lane)[WAVE * i];
#pragma unroll
                for (int e = 0; e < 4; ++e) x[e] = fold_sum(x[e], fa, acc[TR + i][e], fb);
                stot(lane)[WAVE * i] = x;
            }
        }
    };
    clear();
    if constexpr (WALK) {
#pragma unroll
        for (int i = 0; i < TR; ++i) tot[i] = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int i = 0; i < TL; ++i) stot(lane)[WAVE * i] = f32x4_t{0.f, 0.f, 0.f, 0.f};
        if constexpr (TL > 0) *sml(lane) = make_float2(-INFINITY, 0.0f);
    }
    const int vread = (2 * col + v_half(col, jj >> 1)) * 16 + (jj & 1) * 8;   // keys 4 jj .. of row col of a 16-row tile
    const int unit_steps = A.unit / 32;
    int left = unit_steps;   // steps until the unit ends

#pragma unroll
    for (int j = 0; j < S - 1; ++j)
        if (j < nsteps) issue(j);
    for (int i = 0; i < nsteps; ++i) {
        // this wave's loads of step i are done once at most those of the
        // S-2 later steps remain; the barrier makes every wave's loads of
        // step i visible and frees stage (i-1) % S for step i+S-1
        const int later = min(S - 2, nsteps - 1 - i);
        if (later >= 2) wait_loads_barrier<2 * LPW>();
        else if (later == 1) wait_loads_barrier<LPW>();
        else wait_loads_barrier<0>();
        if (i + S - 1 < nsteps) issue(i + S - 1);
        const int kb = k_begin + 32 * i;
        if (kb + 32 > len) {   // the cache ends in this step
            zero_past<D>(lds + (i % S) * St::BYTES + St::K_BYTES, len - kb, TL > 0 ? wave * WAVE + lane_again() : threadIdx.x, 64 * W);
            __syncthreads();
        }
        if (!active || kb > wave_last) continue;   // every key of this step and the later ones is masked
        if (left == 0) {
            unit_end();
            clear();
            left = unit_steps;
        }
        const bool fresh = left == unit_steps;
        --left;
        const char* stage = lds + (i % S) * St::BYTES;
        // ---- S^T for the two 16-key tiles
        f32x4_t sacc[2];
#pragma unroll
        for (int a = 0; a < 2; ++a) {
            sacc[a] = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int st = 0; st < NSTEP; ++st) {
                const bf16x8_t kv = *reinterpret_cast<const bf16x8_t*>(stage + (a * NSTEP + st) * 1024 + lane * 16);
                sacc[a] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kv, qhi[st], sacc[a], 0, 0, 0);
                sacc[a] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(kv, qlo[st], sacc[a], 0, 0, 0);
            }
        }
        // ---- mask, online softmax for this lane's row (keys 4jj+r, 16+4jj+r)
        float p[8];
#pragma unroll
        for (int k = 0; k < 8; ++k) p[k] = sacc[k / 4][k % 4];
        if (kb + 31 > wave_all) {   // some row does not see the whole step
            const int last = last_key(s0, t, len), first = kb + (TL > 0 ? lane_again() / 16 : jj) * 4;
#pragma unroll
            for (int k = 0; k < 8; ++k)
                if (first + 16 * (k / 4) + k % 4 > last) p[k] = -INFINITY;
        }
        float mx = p[0];
#pragma unroll
        for (int k = 1; k < 8; ++k) mx = fmaxf(mx, p[k]);
        const float m_new = fmaxf(m_run, lanegroup_max(mx));
        const float ms = (m_new == -INFINITY) ? 0.0f : m_new;   // a row that sees no key yet: p = 0
        float sum = 0.0f;
#pragma unroll
        for (int k = 0; k < 8; ++k) {
            p[k] = exp2_hw(p[k] - ms);
            sum += p[k];
        }
        // alpha is exactly 1 when the row's max did not move, so the
        // accumulators need rescaling only when some row of the wave moved
        // (and not in a new unit, where they are zero)
        const float alpha = (m_new == m_run) ? 1.0f : exp2_hw(m_run - m_new);
        l_run = l_run * alpha + sum;
        m_run = m_new;
        if (!fresh && __any(alpha != 1.0f)) {
#pragma unroll
            for (int dt = 0; dt < NDT; ++dt) acc[dt] *= alpha;
        }
        bf16x8_t phi, plo;
#pragma unroll
        for (int k = 0; k < 8; k += 2) split_pair(p[k], p[k + 1], phi, plo, k);
        // ---- O^T += V^T . P^T over the 32 keys
        const char* vs = stage + St::K_BYTES;
#pragma unroll
        for (int dt = 0; dt < NDT; ++dt) {
            const uint2 lo2 = *reinterpret_cast<const uint2*>(vs + vread + 512 * dt);
            const uint2 hi2 = *reinterpret_cast<const uint2*>(vs + vread + St::V_BLOCK + 512 * dt);
            const bf16x8_t vv = __builtin_bit_cast(bf16x8_t, uint4{lo2.x, lo2.y, hi2.x, hi2.y});
            acc[dt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(vv, phi, acc[dt], 0, 0, 0);
            acc[dt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(vv, plo, acc[dt], 0, 0, 0);
        }
    }
    if (!active || k_begin > wave_last) return;
    unit_end();
    if constexpr (WALK) {
        const int lane = TL > 0 ? lane_again() : 0;
#pragma unroll
        for (int i = 0; i < NDT; ++i) acc[i] = i < TR ? tot[i] : stot(lane)[WAVE * (i - TR)];
        store(slot0, m_tot, l_tot, acc);
    }
}

// The generic kernel's merge of each query row's chunk partials; chunks that start past the
// row's position were never computed for it and are skipped. The global max
// comes first, so the weighted sums are independent terms: wave w sums
// chunks w, w + 4, ... (lane: channels lane and lane + 64, 8 chunks' loads in
// flight) and the 4 waves' sums meet in LDS in wave order. The result depends
// only on the row's own chunks, never on the batch or the launch shape.
constexpr int PCOMB_WAVES = 4;
__global__ void __launch_bounds__(64 * PCOMB_WAVES) paged_merge_kernel(const float* __restrict__ part, int T,
                                                                         int Hq, int D,
                                                                         const int32_t* __restrict__ start,
                                                                         const int32_t* __restrict__ count, int CH,
                                                                         int n_chunks, float* __restrict__ out) {
    const int hq = blockIdx.x, t = blockIdx.y, s = blockIdx.z;
    // the last key the row saw: its own position, or the cache end for a
    // padding row (t >= count[s]), which attends over the whole cache
    const int len = start[s] + (count ? count[s] : T);
    const int last = min(start[s] + t, len - 1);
    if (last < 0) {   // an empty cache (count 0 at start 0): nothing to attend to
        for (int d = threadIdx.x; d < D; d += blockDim.x) out[(((int64_t)s * T + t) * Hq + hq) * D + d] = 0.0f;
        return;
    }
    const int nc = min(last / CH + 1, n_chunks);   // never past the workspace
    const int PD = D + 2;
    const float* p = part + (((int64_t)s * T + t) * Hq + hq) * n_chunks * PD;
    const int w = threadIdx.x / WAVE, lane = threadIdx.x % WAVE;
    __shared__ float smax[PCOMB_WAVES], sl[PCOMB_WAVES];
    __shared__ float so[PCOMB_WAVES][2 * WAVE];
    float mm = -INFINITY;
    for (int c = threadIdx.x; c < nc; c += blockDim.x) mm = fmaxf(mm, p[(int64_t)c * PD + D]);
    for (int o = WAVE / 2; o > 0; o >>= 1) mm = fmaxf(mm, __shfl_xor(mm, o));
    if (lane == 0) smax[w] = mm;
    __syncthreads();
    mm = smax[0];
#pragma unroll
    for (int i = 1; i < PCOMB_WAVES; ++i) mm = fmaxf(mm, smax[i]);
    const bool a0 = lane < D, a1 = lane + WAVE < D;
    float l = 0.0f, o0 = 0.0f, o1 = 0.0f;
#pragma unroll 8
    for (int c = w; c < nc; c += PCOMB_WAVES) {
        const float* pc = p + (int64_t)c * PD;
        const float mc = pc[D], lc = pc[D + 1];
        const float x0 = a0 ? pc[lane] : 0.0f, x1 = a1 ? pc[lane + WAVE] : 0.0f;
        const float wt = (mc == -INFINITY) ? 0.0f : __expf(mc - mm);
        l = fmaf(lc, wt, l);
        o0 = fmaf(x0, wt, o0);
        o1 = fmaf(x1, wt, o1);
    }
    so[w][lane] = o0;
    so[w][lane + WAVE] = o1;
    if (lane == 0) sl[w] = l;
    __syncthreads();
    for (int d = threadIdx.x; d < D; d += blockDim.x) {
        float lt = 0.0f, ot = 0.0f;
#pragma unroll
        for (int i = 0; i < PCOMB_WAVES; ++i) {
            lt += sl[i];
            ot += so[i][d];
        }
        out[(((int64_t)s * T + t) * Hq + hq) * D + d] = ot / lt;
    }
}

// ------------------------------------------------------------ bf16 path: plan and launch
struct Bf16Shape {
    int W, groups;   // waves (q-tiles) per workgroup, workgroups per (sequence, KV head)
};
// triples: (sequence, KV head, chunk)
static Bf16Shape bf16_shape(int n_qtiles, int64_t triples) {
    Bf16Shape f;
    // one wave per q-tile, up to 8 per workgroup (a power of two, so a step's loads split evenly); a prompt's
    // workgroups take 4 (twice as many of them: 393 against 480 us for 4096 rows)
    f.W = n_qtiles <= 1 ? 1 : n_qtiles <= 2 ? 2 : n_qtiles <= 4 || n_qtiles > 8 ? 4 : 8;
    // Five to eight q-tiles where a workgroup of eight per chunk would leave CUs with one of them, and units, at
    // 66 KB of partials written and read beside 64 KB of K and V, cost more than they spread: two workgroups of
    // four walk each chunk, the second reading from its XCD's L2. Eight waves in units / two groups of four,
    // Llama-3-8B heads, T = 17 / 32, us: batch 1 ctx 64k (256 triples) 112 / 161 -> 104 / 104, batch 2 ctx 48k
    // (384) 162 / 276 -> 130 / 142; below (192: batch 1 ctx 48k) 88 / 125 against 101 / 129, above (512: batch 2
    // ctx 64k, eight waves walking) 136 / 172 against 181 / 195.
    if (f.W == 8 && triples >= 256 && triples < 512) f.W = 4;
    f.groups = (n_qtiles + f.W - 1) / f.W;
    return f;
}

// Slots are chunks when their workgroups fill the chip well enough, or half the
// CUs with one for a prompt's long rows (whose units' partials would be more
// traffic than K and V); else units, so that a single sequence's cache is read
// by more than one workgroup per head, in runs that make one resident round of
// four workgroups per CU. A walk's time hardly depends on how many there are
// up to 512; units' grows with the keys and, by their partials, with the rows.
// Units / chunks, us, Llama-3-8B heads at 256, 320, 384 and 480 chunk
// workgroups (batch 2 ctx 32k and 40k, batch 3 ctx 32k and 40k; a row's merge
// adds about what one more workgroup per chunk does): T = 1 61 / 77,
// 71 / 88, 83 / 92, 108 / 100; T = 5 74 / 82, 90 / 97, 104 / 98, 131 / 100; T =
// 9 83 / 86, 104 / 98, 121 / 100, 151 / 102; T = 13 94 / 89, 124 / 103, 138 /
// 105, 172 / 108; 9 heads on 3 of 64, batch 4 ctx 64k (384), T = 1 / 10 / 20
// 47 / 67, 73 / 69, 96 / 72; 8 on one, batch 3 ctx 262k (384 of 128 chunks), T =
// 1 123 / 103.
// Units' partials take more workspace than chunks', so a smaller call may ask
// for more of it than a larger one: in `work_bytes` that hold no more than the
// chunks' partials, slots are chunks.
static PagedAttnArgs bf16_plan(const dkv_paged_t& c, int T, int Hq, int max_len, int chunk_keys, size_t work_bytes) {
    PagedAttnArgs a = {};
    a.c = c, a.T = T, a.Hq = Hq, a.CH = chunk_keys;
    a.unit = chunk_keys % 128 == 0 ? 128 : chunk_keys % 64 == 0 ? 64 : 32;
    a.n_qtiles = (int)(((int64_t)T * (Hq / c.n_kv_heads) + QB - 1) / QB);
    const int64_t n_chunks = (max_len + chunk_keys - 1) / chunk_keys, n_units = (max_len + a.unit - 1) / a.unit;
    const int64_t pairs = (int64_t)c.n_kv_heads * c.batch;
    const Bf16Shape f = bf16_shape(a.n_qtiles, n_chunks * pairs);
    const bool wide = c.head_dim == 128;
    const int fill = a.n_qtiles > 8 ? 128 : f.W == 4 ? 256 : f.W == 2 ? (wide ? 384 : 448) : f.W == 1 && wide ? 448 : 512;
    const int64_t wgs = f.groups * pairs;
    const bool walk = n_chunks * (wgs + (a.n_qtiles > 8 ? 0 : 1)) >= fill || n_units > 65535 ||
                      work_bytes < paged_part_bytes(c, T, Hq, (int)n_units);
    a.span = walk ? chunk_keys : a.unit;
    a.n_slots = (int)(walk ? n_chunks : n_units);
    a.run = walk ? 1 : (int)((n_units * wgs + 1023) / 1024);
    return a;
}

static bool paged_bf16_takes(const dkv_paged_t& c) {
    return c.dtype == DKV_BF16 && c.block_size == 16 && (c.head_dim == 64 || c.head_dim == 128);
}

static int paged_bf16_attention(const dkv_paged_t& c, int layer, const float* q, int T, int Hq, const int32_t* start,
                                const int32_t* count, int max_len, int chunk_keys, float* out, void* work,
                                size_t work_bytes, hipStream_t st) {
    PagedAttnArgs a = bf16_plan(c, T, Hq, max_len, chunk_keys, work_bytes);
    a.layer = layer, a.q = q, a.start = start, a.count = count, a.out = out;
    a.qscale = static_cast<float>(1.4426950408889634 / sqrt(static_cast<double>(c.head_dim)));
    paged_set_work(a, work);
    const bool walk = a.span == chunk_keys;
    Bf16Shape f = bf16_shape(a.n_qtiles, (int64_t)((max_len + chunk_keys - 1) / chunk_keys) * c.n_kv_heads * c.batch);
    // stages (a unit's four steps all in flight, longer ranges two) and the range's block ids
    const int stages = walk || a.run > 1 ? 2 : 4;
    auto lds_of = [&](int s, int64_t keys) {
        return s * (size_t)(c.head_dim == 128 ? VerifyStage<128>::BYTES : VerifyStage<64>::BYTES) +
               (((size_t)keys / 16 * 4 + 15) & ~size_t(15));
    };
    int fold = fold_bytes(fold_tiles(c.head_dim, f.W, walk, f.groups == 1), f.W);
    bool cached = f.groups > 1;   // more than one workgroup reads a key
    if (fold && lds_of(2, chunk_keys) + fold > 160 * 1024) {   // the ids of a chunk of 390k keys and more leave no room:
        f.W = 4, f.groups = (a.n_qtiles + 3) / 4;              // the form whose sums all stay in registers
        fold = 0, cached = true;
    }
    const size_t lds = lds_of(stages, (int64_t)a.run * a.span) + fold;
    // gfx950 gives a workgroup up to 160 KB of LDS; the chunk must fit whatever this call's ranges are, so that
    // a cache whose chunks some call would not take is refused by every call
    DKV_REQUIRE(lds_of(2, chunk_keys) <= 160 * 1024 && lds <= 160 * 1024,
                "dkv_paged_attention: chunk_keys too large for the bf16 kernel");
    DKV_REQUIRE((int64_t)c.n_kv_heads * c.batch <= 65535 && a.n_slots <= 65535,
                "dkv_paged_attention: batch x heads or chunk count too large for the grid");
    const dim3 blk(64 * f.W);
#define DKV_VERIFY(DD, WW, SS, KK, NN)                                                                             \
    do {                                                                                                           \
        auto kfn = paged_attn_mfma_kernel<DD, WW, SS, KK, NN>;                                                     \
        static size_t lds_done[16] = {};                                                                           \
        if (!reserve_lds(reinterpret_cast<const void*>(kfn), lds, lds_done))                                       \
            return fail(DKV_ELAUNCH, "dkv_paged_attention: cannot reserve " + std::to_string(lds) + " B of LDS");  \
        /* a grid's y holds 65535 q-groups */                                                                      \
        for (a.group0 = 0; a.group0 < f.groups; a.group0 += 65535)                                                 \
            hipLaunchKernelGGL(kfn, dim3(c.n_kv_heads * c.batch, std::min(f.groups - a.group0, 65535),             \
                                         (a.n_slots + a.run - 1) / a.run), blk, lds, st, a);                       \
    } while (0)
#define DKV_VERIFY_W(DD, WW, NN)                        \
    do {                                                \
        if (walk) DKV_VERIFY(DD, WW, 2, true, NN);               \
        else if (a.run > 1) DKV_VERIFY(DD, WW, 2, false, NN);    \
        else DKV_VERIFY(DD, WW, 4, false, NN);                   \
    } while (0)
#define DKV_VERIFY_D(DD)                                \
    do {                                                \
        if (cached) DKV_VERIFY_W(DD, 4, false);         \
        else if (f.W == 8) DKV_VERIFY_W(DD, 8, true);   \
        else if (f.W == 4) DKV_VERIFY_W(DD, 4, true);   \
        else if (f.W == 2) DKV_VERIFY_W(DD, 2, true);   \
        else DKV_VERIFY_W(DD, 1, true);                 \
    } while (0)
    if (c.head_dim == 128) DKV_VERIFY_D(128);
    else DKV_VERIFY_D(64);
#undef DKV_VERIFY_D
#undef DKV_VERIFY_W
#undef DKV_VERIFY
    const int rc = check_launch("dkv_paged_attention");
    return rc || a.n_slots == 1 ? rc : paged_combine(a, st);
}

static size_t attn_smem(int D) {
    return sizeof(float) * (QB * D + KT * (D + 1) + KT * D + QB * KT + 3 * QB);
}

}  // namespace dkv

extern "C" int dkv_paged_append(const dkv_paged_t* cache, int32_t layer, const void* k, const void* v,
                                int32_t in_dtype, int32_t T, const int32_t* start, const int32_t* count,
                                dkv_stream_t stream) {
    DKV_REQUIRE(cache && k && v && start, "dkv_paged_append: NULL argument");
    const dkv_paged_t c = *cache;
    DKV_REQUIRE(layer >= 0 && layer < c.n_layers, "dkv_paged_append: layer out of range");
    DKV_REQUIRE(c.dtype == DKV_F32 || c.dtype == DKV_BF16, "dkv_paged_append: bad cache dtype");
    DKV_REQUIRE(in_dtype == DKV_F32 || in_dtype == DKV_BF16, "dkv_paged_append: bad input dtype");
    DKV_REQUIRE(c.batch > 0 && c.block_size > 0 && c.max_blocks > 0, "dkv_paged_append: bad cache shape");
    if (T <= 0) return DKV_OK;
    // whole blocks for long prompts (paged_append_block_kernel; 16-byte stores of V^T: an aligned pool)
    const int64_t elems = (int64_t)c.batch * T * c.n_kv_heads * c.head_dim;
    if (T >= 64 && elems >= (c.dtype == DKV_F32 ? 200000 : in_dtype == DKV_F32 ? 600000 : 256000) && c.block_size == 16 && reinterpret_cast<uintptr_t>(c.pool) % 16 == 0 && c.batch <= 65535 &&
        c.n_kv_heads <= 65535) {
        const dim3 grid((T + 15) / 16 + 1, c.n_kv_heads, c.batch), blk(c.head_dim <= 64 ? 64 : 128);
#define DKV_APPEND(BB, XX)                                                                                            \
    hipLaunchKernelGGL((dkv::paged_append_block_kernel<BB, XX>), grid, blk, 0, dkv::as_stream(stream), c, layer,      \
                       static_cast<const XX*>(k), static_cast<const XX*>(v), T, start, count)
        if (c.dtype == DKV_BF16 && in_dtype == DKV_BF16) DKV_APPEND(true, uint16_t);
        else if (c.dtype == DKV_BF16) DKV_APPEND(true, float);
        else if (in_dtype == DKV_BF16) DKV_APPEND(false, uint16_t);
        else DKV_APPEND(false, float);
#undef DKV_APPEND
        return dkv::check_launch("dkv_paged_append");
    }
    hipLaunchKernelGGL(dkv::paged_append_kernel, dim3(T, c.batch), dim3(256), 0, dkv::as_stream(stream), c, layer,
                       k, v, in_dtype, T, start, count);
    return dkv::check_launch("dkv_paged_append");
}

static int n_chunks_for(int max_len, int chunk_keys) { return (max_len + chunk_keys - 1) / chunk_keys; }

extern "C" size_t dkv_paged_attention_workspace(const dkv_paged_t* cache, int32_t T, int32_t n_q_heads,
                                                int32_t max_len, int32_t chunk_keys) {
    if (!cache || T <= 0 || n_q_heads <= 0 || max_len <= 0 || chunk_keys <= 0) return 0;
    if (dkv::paged_bf16_takes(*cache))
        return dkv::paged_part_bytes(*cache, T, n_q_heads,
                                     dkv::bf16_plan(*cache, T, n_q_heads, max_len, chunk_keys, SIZE_MAX).n_slots);
    if (dkv::paged_f32_takes(*cache, chunk_keys))
        return dkv::paged_f32_workspace(*cache, T, n_q_heads, max_len, chunk_keys);
    return dkv::paged_part_bytes(*cache, T, n_q_heads, n_chunks_for(max_len, chunk_keys));
}

extern "C" int dkv_paged_attention(const dkv_paged_t* cache, int32_t layer, const float* q, int32_t T,
                                   int32_t n_q_heads, const int32_t* start, const int32_t* count, int32_t max_len,
                                   int32_t chunk_keys, float* out, void* work, size_t work_bytes,
                                   dkv_stream_t stream) {
    DKV_REQUIRE(cache && q && start && out, "dkv_paged_attention: NULL argument");
    const dkv_paged_t c = *cache;
    DKV_REQUIRE(layer >= 0 && layer < c.n_layers, "dkv_paged_attention: layer out of range");
    DKV_REQUIRE(c.head_dim > 0 && c.head_dim <= dkv::MAXD, "dkv_paged_attention: head_dim must be 1..128");
    DKV_REQUIRE(n_q_heads > 0 && n_q_heads % c.n_kv_heads == 0,
                "dkv_paged_attention: query heads must be a multiple of KV heads");
    DKV_REQUIRE(chunk_keys > 0 && chunk_keys % dkv::KT == 0, "dkv_paged_attention: chunk_keys must be a multiple of 32");
    DKV_REQUIRE(max_len > 0, "dkv_paged_attention: max_len must be > 0");
    if (T <= 0) return DKV_OK;
    // one partial per chunk is enough on every path
    const size_t need = dkv::paged_part_bytes(c, T, n_q_heads, n_chunks_for(max_len, chunk_keys));
    if (!work || work_bytes < need)
        return dkv::fail(DKV_EWORKSPACE, "dkv_paged_attention: workspace too small (need " + std::to_string(need) + ")");
    // the kernel choice depends on the cache and its chunks only (never on T or
    // max_len), so a verify pass and a one-token decode step take the same
    // arithmetic path
    if (dkv::paged_bf16_takes(c))
        return dkv::paged_bf16_attention(c, layer, q, T, n_q_heads, start, count, max_len, chunk_keys, out, work,
                                         work_bytes, dkv::as_stream(stream));
    if (dkv::paged_f32_takes(c, chunk_keys))
        return dkv::paged_f32_attention(c, layer, q, T, n_q_heads, start, count, max_len, chunk_keys, out, work,
                                        work_bytes, dkv::as_stream(stream));
    const int n_chunks = n_chunks_for(max_len, chunk_keys);
    const int G = n_q_heads / c.n_kv_heads;
    const int n_qtiles = (T * G + dkv::QB - 1) / dkv::QB;
    DKV_REQUIRE((int64_t)n_chunks * n_qtiles < (1LL << 31), "dkv_paged_attention: grid too large");
    const float scale = static_cast<float>(1.0 / sqrt(static_cast<double>(c.head_dim)));
    hipStream_t st = dkv::as_stream(stream);
    hipLaunchKernelGGL(dkv::paged_attn_kernel, dim3(n_chunks * n_qtiles, c.n_kv_heads, c.batch), dim3(256),
                       dkv::attn_smem(c.head_dim), st, c, layer, q, T, n_q_heads, start, count, chunk_keys,
                       n_chunks, n_qtiles, scale, static_cast<float*>(work));
    int rc = dkv::check_launch("dkv_paged_attention");
    if (rc) return rc;
    hipLaunchKernelGGL(dkv::paged_merge_kernel, dim3(n_q_heads, T, c.batch), dim3(dkv::WAVE * dkv::PCOMB_WAVES), 0, st,
                       static_cast<const float*>(work), T, n_q_heads, c.head_dim, start, count, chunk_keys, n_chunks,
                       out);
    return dkv::check_launch("dkv_paged_attention(combine)");
}

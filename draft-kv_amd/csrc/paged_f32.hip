// Causal attention over the float32 paged full cache on the float32 matrix
// cores. Reference: draftkv/llama.py:202-218 and the gpt2.py/model.py
// equivalents (read + masked softmax attention).
//
// Arithmetic (the same for every launch shape, so a verify row, a prefill row
// and a one-token decode row at one position agree bit for bit): keys are cut
// into units of 64 at absolute positions. A unit's result for a row is
//   m = max of its scores, p = exp(s - m), l = sum p, o = sum p v
// with one chain of v_mfma_f32_16x16x4_f32 per score and per output. Units
// are folded in order inside a chunk of chunk_keys keys, chunks c, c + 4, ...
// are folded in order, and the four classes in order last, all by `fold`.
// Keys a row may not see add exact zeros, and folding such a unit changes
// nothing.
//
// Layout. S^T[16 keys][16 rows] = K . Q^T takes K straight from the cache: in
// the 16-channel group i lane (col, j) holds channels 16 i + 4 j .. + 3 of key
// `col` (one 16-byte load), and its four components are the k-slots of four
// MFMA steps. The accumulator leaves lane (col, j) with keys 4 j .. 4 j + 3 of
// query row `col`: the B operand of O^T += V^T . P^T when step r takes the
// keys 4 j + r, whose V^T operand is component r of one 16-byte load of the
// block's V^T row. So neither K, V nor P passes through LDS.
//
// Bound: decode and verify by latency at small sizes and by HBM at large ones,
// prefill by the matrix cores. Against one workgroup per 2048-key chunk with
// a scalar dot product per score (times of attention plus merge): 8 x 5 rows
// over 4006 keys, 3 KV heads, D = 64: 827 -> 20 us; one row over 1024 keys:
// 395 -> 13.6 us; a 1000-token prompt, 12 heads: 415 -> 55 us.
#include <algorithm>

#include "paged_f32.h"

namespace dkv {

typedef float pf32x4_t __attribute__((ext_vector_type(4)));
typedef float pf32x4u_t __attribute__((ext_vector_type(4), aligned(4)));   // callers' pointers need 4-byte alignment only

constexpr int UNIT = 64;          // keys per unit: four 16-key blocks
constexpr int UT = UNIT / 16;
constexpr int PF_WAVES = 4;
constexpr int COMB_WAVES32 = 4;

// state (m, l, o) folded with a later part (mu, lu, ou): the factors of both
__device__ __forceinline__ float fold_max(float m, float mu, float& a, float& b) {
    const float mn = fmaxf(m, mu);
    a = (m == mn) ? 1.0f : __expf(m - mn);
    b = (mu == mn) ? 1.0f : __expf(mu - mn);
    return mn;
}
__device__ __forceinline__ float fold_sum(float x, float a, float xu, float b) { return fmaf(x, a, __fmul_rn(xu, b)); }

struct PagedF32Args {
    dkv_paged_t c;
    int layer, T, Hq, CH;
    int n_slots;             // key ranges: chunks (WALK) or units
    int n_qtiles;
    const float* q;
    const int32_t* start;
    const int32_t* count;
    float scale;
    float* part;             // o [row][slot][D]; null: the one range's result goes to out
    float2* ml;              // (m, l) [row][slot]
    float* out;
};

// A wave owns 16 query rows (row r -> step r / G, head h G + r % G) of one
// (sequence, KV head) and one key range: a unit, or with WALK the units of a
// chunk in turn. A workgroup is QW row tiles x PF_WAVES / QW ranges: the row
// tiles' K and V loads meet in L1.
template <int D, int QW, bool WALK>
__global__ void __launch_bounds__(64 * PF_WAVES, D == 128 ? 1 : 2) paged_attn_f32_kernel(PagedF32Args A) {
#pragma clang fp contract(off)
    constexpr int NI = D / 16;
    const dkv_paged_t& c = A.c;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / WAVE), lane = threadIdx.x % WAVE;
    const int col = lane % 16, j = lane / 16;
    // the last row tiles see the most keys: they start first
    const int qtile = (int)(gridDim.x - 1 - blockIdx.x) * QW + wave % QW;
    const int h = blockIdx.y % c.n_kv_heads, s = blockIdx.y / c.n_kv_heads;
    const int slot = blockIdx.z * (PF_WAVES / QW) + wave / QW;
    if (qtile >= A.n_qtiles || slot >= A.n_slots) return;
    const int G = A.Hq / c.n_kv_heads, n_rows = A.T * G;
    const int s0 = A.start[s];
    const int len = s0 + (A.count ? A.count[s] : A.T);   // the cache holds positions 0 .. len-1
    const int row = qtile * 16 + col;
    const bool rvalid = row < n_rows;
    const int t = rvalid ? row / G : 0;
    const int hq = h * G + (rvalid ? row % G : 0);
    const int64_t orow = ((int64_t)s * A.T + t) * A.Hq + hq;
    const int span = WALK ? A.CH : UNIT;
    const int k_begin = slot * span;
    const int max_qpos = s0 + (min(qtile * 16 + 16, n_rows) - 1) / G;
    if (k_begin >= len || k_begin > max_qpos) {
        if (!A.part && len <= 0 && rvalid)   // an empty cache: nothing to attend to
            for (int d = 4 * j; d < D; d += 16)
                *reinterpret_cast<pf32x4u_t*>(A.out + orow * D + d) = pf32x4u_t{0.f, 0.f, 0.f, 0.f};
        return;
    }
    const int n_units = (min(min(k_begin + span, len), max_qpos + 1) - k_begin + UNIT - 1) / UNIT;
    const int qpos = s0 + t;

    pf32x4_t qr[NI];
#pragma unroll
    for (int i = 0; i < NI; ++i)
        qr[i] = rvalid ? *reinterpret_cast<const pf32x4u_t*>(A.q + orow * D + 16 * i + 4 * j) : pf32x4_t{0.f, 0.f, 0.f, 0.f};

    const int32_t* btab = c.block_table + ((int64_t)s * c.n_layers + A.layer) * c.max_blocks;
    const float* pool = static_cast<const float*>(c.pool);
    const int64_t bel = paged_block_elems(c);
    const int64_t koff = ((int64_t)h * 16 + col) * D + 4 * j;
    const int64_t voff = (int64_t)c.n_kv_heads * 16 * D + ((int64_t)h * D + col) * 16 + 4 * j;
    const int last_blk = (len - 1) / 16;   // blocks past the cache's end are read as its last one (and masked)
    auto blk_of = [&](int u, int a) {
        return (int64_t)__builtin_amdgcn_readfirstlane(btab[min((k_begin + UNIT * u) / 16 + a, last_blk)]) * bel;
    };
    pf32x4_t kr[UT][NI], vr[UT][NI];
    auto load_k = [&](int u) {
#pragma unroll
        for (int a = 0; a < UT; ++a) {
            const float* p = pool + blk_of(u, a) + koff;
#pragma unroll
            for (int i = 0; i < NI; ++i) kr[a][i] = *reinterpret_cast<const pf32x4u_t*>(p + 16 * i);
        }
    };
    auto load_v = [&](int u) {
#pragma unroll
        for (int a = 0; a < UT; ++a) {
            const float* p = pool + blk_of(u, a) + voff;
#pragma unroll
            for (int i = 0; i < NI; ++i) vr[a][i] = *reinterpret_cast<const pf32x4u_t*>(p + 256 * i);
        }
    };

    float m = -INFINITY, l = 0.0f;
    pf32x4_t o[NI];
#pragma unroll
    for (int i = 0; i < NI; ++i) o[i] = pf32x4_t{0.f, 0.f, 0.f, 0.f};
    load_k(0);
    load_v(0);
    for (int u = 0; u < n_units; ++u) {
        const int kb = k_begin + UNIT * u;
        pf32x4_t sc[UT];
#pragma unroll
        for (int a = 0; a < UT; ++a) sc[a] = pf32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int i = 0; i < NI; ++i)
#pragma unroll
            for (int e = 0; e < 4; ++e)
#pragma unroll
                for (int a = 0; a < UT; ++a)
                    sc[a] = __builtin_amdgcn_mfma_f32_16x16x4f32(kr[a][i][e], qr[i][e], sc[a], 0, 0, 0);
        if (WALK && u + 1 < n_units) load_k(u + 1);   // in flight behind the softmax and PV of this unit
        // keys 16 a + 4 j + r of this lane's row
        float mu = -INFINITY;
#pragma unroll
        for (int a = 0; a < UT; ++a)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const int key = kb + 16 * a + 4 * j + r;
                sc[a][r] = (rvalid && key <= qpos && key < len) ? sc[a][r] * A.scale : -INFINITY;
                mu = fmaxf(mu, sc[a][r]);
            }
        mu = fmaxf(mu, __shfl_xor(mu, 16));
        mu = fmaxf(mu, __shfl_xor(mu, 32));
        float lu = 0.0f;
#pragma unroll
        for (int a = 0; a < UT; ++a)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                sc[a][r] = (sc[a][r] == -INFINITY) ? 0.0f : __expf(sc[a][r] - mu);
                lu += sc[a][r];
            }
        lu += __shfl_xor(lu, 16);
        lu += __shfl_xor(lu, 32);
        if (kb + UNIT > len) {   // stale rows past the cache's end: 0 * NaN would be NaN
#pragma unroll
            for (int a = 0; a < UT; ++a)
#pragma unroll
                for (int i = 0; i < NI; ++i)
#pragma unroll
                    for (int r = 0; r < 4; ++r)
                        if (kb + 16 * a + 4 * j + r >= len) vr[a][i][r] = 0.0f;
        }
        pf32x4_t ou[NI];
#pragma unroll
        for (int i = 0; i < NI; ++i) ou[i] = pf32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int a = 0; a < UT; ++a)
#pragma unroll
            for (int r = 0; r < 4; ++r)
#pragma unroll
                for (int i = 0; i < NI; ++i)
                    ou[i] = __builtin_amdgcn_mfma_f32_16x16x4f32(vr[a][i][r], sc[a][r], ou[i], 0, 0, 0);
        if constexpr (WALK) {
            if (u + 1 < n_units) load_v(u + 1);
            float fa, fb;
            m = fold_max(m, mu, fa, fb);
            l = fold_sum(l, fa, lu, fb);
#pragma unroll
            for (int i = 0; i < NI; ++i)
#pragma unroll
                for (int e = 0; e < 4; ++e) o[i][e] = fold_sum(o[i][e], fa, ou[i][e], fb);
        } else {
            m = mu;
            l = lu;
#pragma unroll
            for (int i = 0; i < NI; ++i) o[i] = ou[i];
        }
    }
    if (!rvalid) return;
    // lane holds channels 16 i + 4 j .. + 3 of its row
    if (A.part) {
        const int64_t ps = orow * A.n_slots + slot;
#pragma unroll
        for (int i = 0; i < NI; ++i) *reinterpret_cast<pf32x4u_t*>(A.part + ps * D + 16 * i + 4 * j) = o[i];
        if (j == 0) A.ml[ps] = make_float2(m, l);
    } else {
#pragma unroll
        for (int i = 0; i < NI; ++i)
            *reinterpret_cast<pf32x4u_t*>(A.out + orow * D + 16 * i + 4 * j) =
                pf32x4u_t{o[i][0] / l, o[i][1] / l, o[i][2] / l, o[i][3] / l};
    }
}

// Fold a row's ranges: wave w the chunks w, w + 4, ..., a chunk's units (one
// when the ranges are chunks) in order, then the waves in order. Lane:
// channels lane and lane + 64; a batch of units' loads is in flight at once.
__global__ void __launch_bounds__(64 * COMB_WAVES32) paged_combine_f32_kernel(PagedF32Args A, int D, int units) {
    constexpr int NB = 16;   // units per batch of loads
    const int hq = blockIdx.x, t = blockIdx.y, s = blockIdx.z;
    const int s0 = A.start[s], len = s0 + (A.count ? A.count[s] : A.T);
    const int last = min(s0 + t, len - 1);   // a padding row (t >= count) attends over the whole cache
    const int64_t row = ((int64_t)s * A.T + t) * A.Hq + hq;
    if (last < 0) {   // an empty cache: nothing to attend to
        for (int d = threadIdx.x; d < D; d += blockDim.x) A.out[row * D + d] = 0.0f;
        return;
    }
    const int n_live = min(last / (units > 1 ? UNIT : A.CH) + 1, A.n_slots);
    const int w = threadIdx.x / WAVE, lane = threadIdx.x % WAVE;
    const float* po = A.part + row * A.n_slots * D;
    const float2* pm = A.ml + row * A.n_slots;
    const int c0 = min(lane, D - 1), c1 = min(lane + WAVE, D - 1);
    float m = -INFINITY, l = 0.0f, o0 = 0.0f, o1 = 0.0f;
    for (int ck = w; ck * units < n_live; ck += COMB_WAVES32) {
        const int ub = ck * units, ue = min(ub + units, n_live);
        float cm = -INFINITY, cl = 0.0f, x0 = 0.0f, x1 = 0.0f;
        for (int u0 = ub; u0 < ue; u0 += NB) {
            float2 v[NB];
            float y0[NB], y1[NB];
#pragma unroll
            for (int k = 0; k < NB; ++k) {
                const int u = min(u0 + k, ue - 1);
                v[k] = pm[u];
                y0[k] = po[(int64_t)u * D + c0];
                y1[k] = D > WAVE ? po[(int64_t)u * D + c1] : 0.0f;
            }
#pragma unroll
            for (int k = 0; k < NB; ++k) {
                if (u0 + k < ue) {
                    float a, b;
                    cm = fold_max(cm, v[k].x, a, b);
                    cl = fold_sum(cl, a, v[k].y, b);
                    x0 = fold_sum(x0, a, y0[k], b);
                    x1 = fold_sum(x1, a, y1[k], b);
                }
            }
        }
        float a, b;
        m = fold_max(m, cm, a, b);
        l = fold_sum(l, a, cl, b);
        o0 = fold_sum(o0, a, x0, b);
        o1 = fold_sum(o1, a, x1, b);
    }
    __shared__ float sm[COMB_WAVES32], sl[COMB_WAVES32], so[COMB_WAVES32][2 * WAVE];
    so[w][lane] = o0;
    so[w][lane + WAVE] = o1;
    if (lane == 0) sm[w] = m, sl[w] = l;
    __syncthreads();
    for (int d = threadIdx.x; d < D; d += blockDim.x) {
        float rm = sm[0], rl = sl[0], ro = so[0][d];
#pragma unroll
        for (int i = 1; i < COMB_WAVES32; ++i) {
            float a, b;
            rm = fold_max(rm, sm[i], a, b);
            rl = fold_sum(rl, a, sl[i], b);
            ro = fold_sum(ro, a, so[i][d], b);
        }
        A.out[row * D + d] = ro / rl;
    }
}

bool paged_f32_takes(const dkv_paged_t& c, int max_len, int chunk_keys) {
    return c.dtype == DKV_F32 && c.block_size == 16 && chunk_keys % UNIT == 0 &&
           (int64_t)c.n_kv_heads * c.batch <= 65535 && (max_len + UNIT - 1) / UNIT <= 65535 &&
           (c.head_dim == 16 || c.head_dim == 32 || c.head_dim == 64 || c.head_dim == 128);
}

// A wave per (row tile, unit), or, where the (row tile, chunk) pairs alone
// fill half of the chip's 1024 SIMDs, one per pair that walks its units and
// writes one partial per chunk, or the output itself when there is one chunk
// (below that, units in parallel finish sooner than the longest walk: one row
// per sequence would be a chain of up to 32 units on a handful of waves). The
// results are the same bits.
struct PagedF32Plan {
    int n_qtiles, n_slots, units;   // units per chunk when the slots are units, else 1
    bool walk;
};
static PagedF32Plan f32_plan(const dkv_paged_t& c, int T, int Hq, int max_len, int chunk_keys) {
    PagedF32Plan p;
    p.n_qtiles = (int)(((int64_t)T * (Hq / c.n_kv_heads) + 15) / 16);
    const int n_chunks = (max_len + chunk_keys - 1) / chunk_keys;
    p.walk = (int64_t)n_chunks * p.n_qtiles * c.n_kv_heads * c.batch >= 512;
    p.n_slots = p.walk ? n_chunks : (max_len + UNIT - 1) / UNIT;
    p.units = p.walk ? 1 : chunk_keys / UNIT;
    return p;
}

size_t paged_f32_workspace(const dkv_paged_t& c, int T, int Hq, int max_len, int chunk_keys) {
    const PagedF32Plan p = f32_plan(c, T, Hq, max_len, chunk_keys);
    return sizeof(float) * (size_t)c.batch * T * Hq * p.n_slots * (c.head_dim + 2);
}

int paged_f32_attention(const dkv_paged_t& c, int layer, const float* q, int T, int Hq, const int32_t* start,
                        const int32_t* count, int max_len, int chunk_keys, float* out, void* work, hipStream_t stream) {
    const PagedF32Plan p = f32_plan(c, T, Hq, max_len, chunk_keys);
    const int D = c.head_dim;
    const bool direct = p.walk && p.n_slots == 1;
    const int64_t rows = (int64_t)c.batch * T * Hq;
    PagedF32Args a;
    a.c = c, a.layer = layer, a.T = T, a.Hq = Hq, a.CH = chunk_keys, a.n_slots = p.n_slots, a.n_qtiles = p.n_qtiles;
    a.q = q, a.start = start, a.count = count, a.out = out;
    a.scale = static_cast<float>(1.0 / sqrt(static_cast<double>(D)));
    a.part = direct ? nullptr : static_cast<float*>(work);
    a.ml = direct ? nullptr : reinterpret_cast<float2*>(static_cast<float*>(work) + rows * p.n_slots * D);
    const int QW = p.n_qtiles >= 4 ? 4 : p.n_qtiles >= 2 ? 2 : 1;
    const int64_t gx = (p.n_qtiles + QW - 1) / QW, gz = (p.n_slots + PF_WAVES / QW - 1) / (PF_WAVES / QW);
    const dim3 grid((unsigned)gx, c.n_kv_heads * c.batch, (unsigned)gz), blk(64 * PF_WAVES);
#define DKV_PF(DD, QQ)                                                                                       \
    do {                                                                                                     \
        if (p.walk) hipLaunchKernelGGL((paged_attn_f32_kernel<DD, QQ, true>), grid, blk, 0, stream, a);      \
        else hipLaunchKernelGGL((paged_attn_f32_kernel<DD, QQ, false>), grid, blk, 0, stream, a);            \
    } while (0)
#define DKV_PFQ(DD)                     \
    do {                                \
        if (QW == 4) DKV_PF(DD, 4);     \
        else if (QW == 2) DKV_PF(DD, 2); \
        else DKV_PF(DD, 1);             \
    } while (0)
    switch (D) {
        case 16: DKV_PFQ(16); break;
        case 32: DKV_PFQ(32); break;
        case 64: DKV_PFQ(64); break;
        default: DKV_PFQ(128); break;
    }
#undef DKV_PFQ
#undef DKV_PF
    int rc = check_launch("dkv_paged_attention");
    if (rc || direct) return rc;
    hipLaunchKernelGGL(paged_combine_f32_kernel, dim3(Hq, T, c.batch), dim3(64 * COMB_WAVES32), 0, stream, a, D, p.units);
    return check_launch("dkv_paged_attention(combine)");
}

}  // namespace dkv

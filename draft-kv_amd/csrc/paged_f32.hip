// Causal attention over the float32 paged full cache on the float32 matrix
// cores. Reference: draftkv/llama.py:202-218 and the gpt2.py/model.py
// equivalents (read + masked softmax attention).
//
// Units of 64 keys (paged_attn.h); per unit one chain of
// v_mfma_f32_16x16x4_f32 per score and per output.
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
// over 4006 keys, 3 KV heads, D = 64: 827 -> 22 us; one row over 1024 keys:
// 395 -> 13.6 us; a 1000-token prompt, 12 heads: 415 -> 55 us.
#include <algorithm>

#include "paged_attn.h"

namespace dkv {

typedef float pf32x4_t __attribute__((ext_vector_type(4)));
typedef float pf32x4u_t __attribute__((ext_vector_type(4), aligned(4)));   // callers' pointers need 4-byte alignment only

constexpr int UNIT = 64;          // keys per unit: four 16-key blocks
constexpr int UT = UNIT / 16;
constexpr int PF_WAVES = 4;       // per workgroup

// A wave owns 16 query rows (row r -> step r / G, head h G + r % G) of one
// (sequence, KV head) and one key range: a unit, or with WALK the units of a
// chunk in turn. A workgroup is QW row tiles x PF_WAVES / QW ranges: the row
// tiles' K and V loads meet in L1.
template <int D, int QW, bool WALK>
__global__ void __launch_bounds__(64 * PF_WAVES, D == 128 ? 1 : 2) paged_attn_f32_kernel(PagedAttnArgs A) {
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
    const int s0 = __builtin_amdgcn_readfirstlane(A.start[s]);
    const int len = s0 + (A.count ? __builtin_amdgcn_readfirstlane(A.count[s]) : A.T);   // the cache holds positions 0 .. len-1
    const int row = qtile * 16 + col;
    const bool rvalid = row < n_rows;
    const int t = rvalid ? row / G : 0;
    const int hq = h * G + (rvalid ? row % G : 0);
    const int64_t orow = ((int64_t)s * A.T + t) * A.Hq + hq;
    const int k_begin = slot * A.span;
    const int max_qpos = s0 + (min(qtile * 16 + 16, n_rows) - 1) / G;
    if (k_begin >= len || k_begin > max_qpos) {
        if (slot == 0 && len <= 0 && rvalid)   // an empty cache: nothing to attend to
            for (int d = 4 * j; d < D; d += 16)
                *reinterpret_cast<pf32x4u_t*>(A.out + orow * D + d) = pf32x4u_t{0.f, 0.f, 0.f, 0.f};
        return;
    }
    const int n_units = (min(min(k_begin + A.span, len), max_qpos + 1) - k_begin + UNIT - 1) / UNIT;
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
                sc[a][r] = (rvalid && key <= qpos && key < len) ? sc[a][r] * A.qscale : -INFINITY;
                mu = fmaxf(mu, sc[a][r]);
            }
        mu = fmaxf(mu, __shfl_xor(mu, 16));
        mu = fmaxf(mu, __shfl_xor(mu, 32));
        const float ms = (mu == -INFINITY) ? 0.0f : mu;   // a row that sees none of the unit: p = 0
        float lu = 0.0f;
#pragma unroll
        for (int a = 0; a < UT; ++a)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                sc[a][r] = exp2_hw(sc[a][r] - ms);
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
    if (last_key(s0, t, len) >= A.span && A.n_slots > 1) {
        const int64_t ps = orow * A.n_slots + slot;
#pragma unroll
        for (int i = 0; i < NI; ++i) *reinterpret_cast<pf32x4u_t*>(A.part + ps * D + 16 * i + 4 * j) = o[i];
        if (j == 0) A.ml[ps] = make_float2(m, l);
    } else if (slot == 0) {   // the row sees no other slot
#pragma unroll
        for (int i = 0; i < NI; ++i)
            *reinterpret_cast<pf32x4u_t*>(A.out + orow * D + 16 * i + 4 * j) =
                pf32x4u_t{o[i][0] / l, o[i][1] / l, o[i][2] / l, o[i][3] / l};
    }
}

constexpr int MAX_SLOTS = 65535;   // the grid's z

bool paged_f32_takes(const dkv_paged_t& c, int chunk_keys) {
    // (a sequence's chunks fit the grid; calls of more units walk them)
    return c.dtype == DKV_F32 && c.block_size == 16 && chunk_keys % UNIT == 0 &&
           (int64_t)c.n_kv_heads * c.batch <= 65535 && (int64_t)c.max_blocks * 16 <= (int64_t)MAX_SLOTS * chunk_keys &&
           (c.head_dim == 16 || c.head_dim == 32 || c.head_dim == 64 || c.head_dim == 128);
}

// Slots are chunks from 512 (row tile, chunk) pairs on, half of the chip's
// 1024 SIMDs: below that, units in parallel finish sooner than the longest
// walk (one row per sequence would be a chain of up to 32 units on a handful
// of waves). So are they where `work_bytes` hold no more than the chunks'
// partials (a smaller call may ask for more than a larger one).
static PagedAttnArgs f32_plan(const dkv_paged_t& c, int T, int Hq, int max_len, int chunk_keys, size_t work_bytes) {
    PagedAttnArgs a = {};
    a.c = c, a.T = T, a.Hq = Hq, a.CH = chunk_keys, a.unit = UNIT;
    a.n_qtiles = (int)(((int64_t)T * (Hq / c.n_kv_heads) + 15) / 16);
    const int64_t keys = std::min<int64_t>(max_len, (int64_t)c.max_blocks * 16);   // no sequence holds more
    const int64_t n_chunks = (keys + chunk_keys - 1) / chunk_keys, n_units = (keys + UNIT - 1) / UNIT;
    const bool walk = n_units > MAX_SLOTS || n_chunks * a.n_qtiles * c.n_kv_heads * c.batch >= 512 ||
                      work_bytes < paged_part_bytes(c, T, Hq, (int)n_units);
    a.span = walk ? chunk_keys : UNIT;
    a.n_slots = (int)(walk ? n_chunks : n_units);
    return a;
}

size_t paged_f32_workspace(const dkv_paged_t& c, int T, int Hq, int max_len, int chunk_keys) {
    return paged_part_bytes(c, T, Hq, f32_plan(c, T, Hq, max_len, chunk_keys, SIZE_MAX).n_slots);
}

int paged_f32_attention(const dkv_paged_t& c, int layer, const float* q, int T, int Hq, const int32_t* start,
                        const int32_t* count, int max_len, int chunk_keys, float* out, void* work,
                        size_t work_bytes, hipStream_t stream) {
    PagedAttnArgs a = f32_plan(c, T, Hq, max_len, chunk_keys, work_bytes);
    const int D = c.head_dim;
    a.layer = layer, a.q = q, a.start = start, a.count = count, a.out = out;
    a.qscale = static_cast<float>(1.4426950408889634 / sqrt(static_cast<double>(D)));
    paged_set_work(a, work);
    const bool walk = a.span == chunk_keys;
    const int QW = a.n_qtiles >= 4 ? 4 : a.n_qtiles >= 2 ? 2 : 1;
    const int64_t gx = (a.n_qtiles + QW - 1) / QW, gz = (a.n_slots + PF_WAVES / QW - 1) / (PF_WAVES / QW);
    const dim3 grid((unsigned)gx, c.n_kv_heads * c.batch, (unsigned)gz), blk(64 * PF_WAVES);
#define DKV_PF(DD, QQ)                                                                                       \
    do {                                                                                                     \
        if (walk) hipLaunchKernelGGL((paged_attn_f32_kernel<DD, QQ, true>), grid, blk, 0, stream, a);      \
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
    const int rc = check_launch("dkv_paged_attention");
    return rc || a.n_slots == 1 ? rc : paged_combine(a, stream);
}

}  // namespace dkv

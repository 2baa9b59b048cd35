// Folds the slots of dkv_paged_attention's rows (paged_attn.h).
// Reference: the softmax normalisation of draftkv/llama.py:202-218.
#include "paged_attn.h"

namespace dkv {

constexpr int COMB_WAVES4 = 4;

// Slots u0, u0 + step, ... below ue folded into f in order; the lane's channels
// are c0 and c1. NB slots' loads are in flight at once.
struct FoldState {
    float m, l, o0, o1;
};
template <int NB>
__device__ __forceinline__ void fold_slots(FoldState& f, const float* po, const float2* pm, int u0, int step, int ue,
                                           int D, int c0, int c1, bool two) {
    for (; u0 < ue; u0 += NB * step) {
        float2 v[NB];
        float y0[NB], y1[NB];
#pragma unroll
        for (int k = 0; k < NB; ++k) {
            const int u = min(u0 + k * step, ue - 1);
            v[k] = pm[u];
            y0[k] = po[(int64_t)u * D + c0];
            y1[k] = two ? po[(int64_t)u * D + c1] : 0.0f;
        }
#pragma unroll
        for (int k = 0; k < NB; ++k)
            if (u0 + k * step < ue) {
                float a, b;
                f.m = fold_max(f.m, v[k].x, a, b);
                f.l = fold_sum(f.l, a, v[k].y, b);
                f.o0 = fold_sum(f.o0, a, y0[k], b);
                f.o1 = fold_sum(f.o1, a, y1[k], b);
            }
    }
}
__device__ __forceinline__ void fold_into(FoldState& s, const FoldState& f) {
    float a, b;
    s.m = fold_max(s.m, f.m, a, b);
    s.l = fold_sum(s.l, a, f.l, b);
    s.o0 = fold_sum(s.o0, a, f.o0, b);
    s.o1 = fold_sum(s.o1, a, f.o1, b);
}

// The units of chunk ck in order.
__device__ __forceinline__ FoldState fold_chunk(const float* po, const float2* pm, int ck, int per, int n_live, int D,
                                                int c0, int c1, bool two) {
    FoldState g = {-INFINITY, 0.0f, 0.0f, 0.0f};
    const int ue = min((ck + 1) * per, n_live);
    if (ue - ck * per > 4) fold_slots<16>(g, po, pm, ck * per, 1, ue, D, c0, c1, two);
    else fold_slots<4>(g, po, pm, ck * per, 1, ue, D, c0, c1, two);
    return g;
}

// One class of a row's chunks, ck0, ck0 + 4, ...: slots that are chunks are
// folded as they are (folding one into the empty state changes nothing), else
// each chunk's `per` units first.
__device__ __forceinline__ FoldState fold_class(const float* po, const float2* pm, int ck0, int per, int n_live, int D,
                                                int c0, int c1, bool two) {
    const FoldState none = {-INFINITY, 0.0f, 0.0f, 0.0f};
    FoldState f = none;
    if (per == 1) {
        // many chunks: 16 loads in flight (batch 1 ctx 262k, 128 chunks, one row: a call 176 -> 171 us)
        if (n_live > 16) fold_slots<16>(f, po, pm, ck0, COMB_WAVES4, n_live, D, c0, c1, two);
        else if (ck0 + COMB_WAVES4 < n_live) fold_slots<4>(f, po, pm, ck0, COMB_WAVES4, n_live, D, c0, c1, two);
        else fold_slots<1>(f, po, pm, ck0, COMB_WAVES4, n_live, D, c0, c1, two);
        return f;
    }
    for (int ck = ck0; ck * per < n_live; ck += COMB_WAVES4)
        fold_into(f, fold_chunk(po, pm, ck, per, n_live, D, c0, c1, two));
    return f;
}

// Grid (query heads, rows, sequences). MANY: one wave per row takes the four
// chunk classes in turn and four rows share a workgroup (a prompt: rows are
// plenty and see few chunks); else the waves share a row. Four of them take
// one class each; sixteen (CHUNKS, for slots that are units) a chunk each and
// round, whose states the first four fold: a class alone is a serial chain of
// its chunks' loads, half a microsecond per chunk of the row (batch 2 ctx 131k,
// 9 heads on 3 of 64, 64 chunks, one row: a call 72 -> 57 us). Sixteen waves
// per row pay while the rows are few, up to eight per chunk (batch 3 ctx 40k,
// 20 chunks, 32 heads, 13 rows: 172 / 184).
constexpr int CHUNK_WAVES = 16;
template <bool MANY, bool CHUNKS>
__global__ void __launch_bounds__(64 * (CHUNKS ? CHUNK_WAVES : COMB_WAVES4)) paged_combine_kernel(PagedAttnArgs A) {
    const int w = __builtin_amdgcn_readfirstlane(threadIdx.x / WAVE), lane = threadIdx.x % WAVE;
    const int D = A.c.head_dim, s = blockIdx.z;
    const int hq = blockIdx.x, t = MANY ? blockIdx.y * COMB_WAVES4 + w : blockIdx.y;
    if (MANY && t >= A.T) return;
    const int s0 = A.start[s], len = s0 + (A.count ? A.count[s] : A.T);
    const int last = last_key(s0, t, len);
    const int n_live = last < 0 ? 0 : min(last / A.span + 1, A.n_slots);   // never past the workspace
    if (n_live <= 1) return;                                               // the attention kernel wrote the row
    const int64_t row = ((int64_t)s * A.T + t) * A.Hq + hq;
    const float* po = A.part + row * A.n_slots * D;
    const float2* pm = A.ml + row * A.n_slots;
    const int per = A.CH / A.span;   // slots per chunk
    const int c0 = min(lane, D - 1), c1 = min(lane + WAVE, D - 1);
    const bool two = D > WAVE;
    FoldState tot;
    if constexpr (MANY) {
        tot = fold_class(po, pm, 0, per, n_live, D, c0, c1, two);
        for (int k = 1; k < COMB_WAVES4; ++k) fold_into(tot, fold_class(po, pm, k, per, n_live, D, c0, c1, two));
    } else {
        __shared__ FoldState sf[CHUNKS ? CHUNK_WAVES : COMB_WAVES4][WAVE];
        FoldState f = {-INFINITY, 0.0f, 0.0f, 0.0f};
        if constexpr (CHUNKS) {
            const int n_chunks = (n_live + per - 1) / per;
            for (int base = 0; base < n_chunks; base += CHUNK_WAVES) {
                if (base + w < n_chunks) sf[w][lane] = fold_chunk(po, pm, base + w, per, n_live, D, c0, c1, two);
                __syncthreads();
                if (w < COMB_WAVES4)
                    for (int i = w; i < CHUNK_WAVES && base + i < n_chunks; i += COMB_WAVES4) fold_into(f, sf[i][lane]);
                __syncthreads();
            }
        } else {
            f = fold_class(po, pm, w, per, n_live, D, c0, c1, two);
        }
        if (w < COMB_WAVES4) sf[w][lane] = f;
        __syncthreads();
        if (w != 0) return;
        tot = sf[0][lane];
#pragma unroll
        for (int k = 1; k < COMB_WAVES4; ++k) fold_into(tot, sf[k][lane]);
    }
    if (lane < D) A.out[row * D + lane] = tot.o0 / tot.l;
    if (lane + WAVE < D) A.out[row * D + lane + WAVE] = tot.o1 / tot.l;
}

size_t paged_part_bytes(const dkv_paged_t& c, int T, int Hq, int n_slots) {
    return sizeof(float) * (size_t)c.batch * T * Hq * n_slots * (c.head_dim + 2);
}

void paged_set_work(PagedAttnArgs& a, void* work) {
    a.part = static_cast<float*>(work);
    a.ml = reinterpret_cast<float2*>(a.part + ((int64_t)a.c.batch * a.T * a.Hq * a.n_slots * a.c.head_dim + 1) / 2 * 2);
}

int paged_combine(const PagedAttnArgs& a, hipStream_t stream) {
    const int64_t rows = (int64_t)a.Hq * a.T * a.c.batch;
    const int64_t chunks = a.span < a.CH ? (int64_t)a.n_slots * a.span / a.CH : 0;   // where slots are units
    // from 64 rows per sequence on, a wave per row: a 4096-token prompt's rows, 32 heads
    if (a.T >= 64)
        hipLaunchKernelGGL((paged_combine_kernel<true, false>), dim3(a.Hq, (a.T + COMB_WAVES4 - 1) / COMB_WAVES4, a.c.batch),
                           dim3(64 * COMB_WAVES4), 0, stream, a);
    else if (chunks > 4 && rows <= 8 * chunks)
        hipLaunchKernelGGL((paged_combine_kernel<false, true>), dim3(a.Hq, a.T, a.c.batch), dim3(64 * CHUNK_WAVES), 0, stream, a);
    else
        hipLaunchKernelGGL((paged_combine_kernel<false, false>), dim3(a.Hq, a.T, a.c.batch), dim3(64 * COMB_WAVES4), 0, stream, a);
    return check_launch("dkv_paged_attention(combine)");
}

}  // namespace dkv

// What the two matrix-core paths of dkv_paged_attention share: the bf16 cache
// (paged.hip) and the float32 one (paged_f32.hip).
//
// Arithmetic (the same for every launch shape, so a verify row, a prompt's
// row and a one-token decode row at one position agree bit for bit): keys are
// cut into units at absolute positions, each unit's softmax state of a row
// (m, l, o: base-2 score maximum, sum of 2^(s - m), weighted sum of V) is
// computed on its own, a chunk's units are folded in order, the chunks
// c, c + 4, ... are folded in order, and these four classes in order last, all
// by fold_max / fold_sum. Keys a row may not see add exact zeros, and folding
// a unit of such keys changes nothing.
//
// A launch computes a row's state over ranges of keys ("slots"): one unit
// each, or, where the (query rows, chunk) pairs alone fill the chip, one
// chunk each, whose units a wave folds as it walks them. The combine kernel
// folds the slots; a row whose keys lie in the first slot is written by the
// attention kernel itself. The host knows max_len, not the sequences'
// lengths: n_slots are the slots that max_len reaches into, no slot past them
// is written and no key past them read, whatever start + count say.
#pragma once

#include "dkv_common.h"

namespace dkv {

struct PagedAttnArgs {
    dkv_paged_t c;
    int layer, T, Hq;
    int CH;                  // keys per chunk
    int unit;                // keys per unit; CH is a multiple of it
    int span;                // keys per slot: CH or unit
    int run;                 // consecutive slots per workgroup (bf16 path)
    int group0;              // the launch's first q-group (bf16 path)
    int n_slots, n_qtiles;
    const float* q;
    const int32_t* start;
    const int32_t* count;
    float qscale;            // log2(e) / sqrt(head_dim): scores are base-2 exponents
    float* part;             // o [row][slot][D]
    float2* ml;              // (m, l) [row][slot]
    float* out;
};

__device__ __forceinline__ float exp2_hw(float x) { return __builtin_amdgcn_exp2f(x); }

// state (m, l, o) folded with a later part (mu, lu, ou): the new m and the factors of both
__device__ __forceinline__ float fold_max(float m, float mu, float& a, float& b) {
    const float mn = fmaxf(m, mu);
    a = (m == mn) ? 1.0f : exp2_hw(m - mn);
    b = (mu == mn) ? 1.0f : exp2_hw(mu - mn);
    return mn;
}
__device__ __forceinline__ float fold_sum(float x, float a, float xu, float b) { return fmaf(x, a, __fmul_rn(xu, b)); }

// The largest key of row t of a sequence: its own position, or the cache's
// last for a padding row (t >= count), which attends over the whole cache;
// -1 for an empty cache.
__device__ __forceinline__ int last_key(int s0, int t, int len) { return min(s0 + t, len - 1); }

// bytes of the partial section, and the slots' pointers in the workspace
size_t paged_part_bytes(const dkv_paged_t& c, int T, int Hq, int n_slots);
void paged_set_work(PagedAttnArgs& a, void* work);
int paged_combine(const PagedAttnArgs& a, hipStream_t stream);

// float32 caches in 16-token blocks, head_dim 16, 32, 64 or 128, chunks of whole 64-key units, sizes within the
// launch grid. A function of the cache and its chunks alone: the generic kernel's rows differ in their last bits,
// so every call on one cache takes the same kernel.
bool paged_f32_takes(const dkv_paged_t& c, int chunk_keys);
size_t paged_f32_workspace(const dkv_paged_t& c, int T, int Hq, int max_len, int chunk_keys);
int paged_f32_attention(const dkv_paged_t& c, int layer, const float* q, int T, int Hq, const int32_t* start,
                        const int32_t* count, int max_len, int chunk_keys, float* out, void* work,
                        size_t work_bytes, hipStream_t stream);

}  // namespace dkv

// The float32 full cache's attention path (paged_f32.hip), behind
// dkv_paged_attention / dkv_paged_attention_workspace (paged.hip).
#pragma once

#include "dkv_common.h"

namespace dkv {

// float32 caches in 16-token blocks, head_dim 16, 32, 64 or 128, key chunks of whole 64-key units
// (and sizes within the launch grid)
bool paged_f32_takes(const dkv_paged_t& c, int max_len, int chunk_keys);
size_t paged_f32_workspace(const dkv_paged_t& c, int T, int Hq, int max_len, int chunk_keys);
int paged_f32_attention(const dkv_paged_t& c, int layer, const float* q, int T, int Hq, const int32_t* start,
                        const int32_t* count, int max_len, int chunk_keys, float* out, void* work,
                        hipStream_t stream);

}  // namespace dkv

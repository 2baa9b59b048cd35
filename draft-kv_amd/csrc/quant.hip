// Group quantizer on contiguous rows -- reference draftkv/compress.py:21-46.
#include "dkv_common.h"

namespace dkv {

// One wave per row; the wave walks the row's groups. Lane l of a group covers
// elements l, l+64, ... of it; elements past d are the zero padding the
// reference appends (compress.py:32-35), which joins the last group's min/max.
__global__ void __launch_bounds__(256) quantize_rows_kernel(const float* __restrict__ x, int64_t rows, int d,
                                                            int bits, int group, int meta_f16,
                                                            uint8_t* codes, float* scale, float* lo,
                                                            float* deq) {
    const int lane = threadIdx.x % WAVE;
    const int64_t row = (int64_t)blockIdx.x * (blockDim.x / WAVE) + threadIdx.x / WAVE;
    if (row >= rows) return;
    const float* xr = x + row * d;
    const int ng = n_groups(d, group);
    for (int g = 0; g < ng; ++g) {
        float mn = INFINITY, mx = -INFINITY;
        for (int e = lane; e < group; e += WAVE) {
            const int j = g * group + e;
            const float v = j < d ? xr[j] : 0.0f;
            mn = fminf(mn, v);
            mx = fmaxf(mx, v);
        }
        mn = wave_min(mn);
        mx = wave_max(mx);
        const GroupMeta m = group_meta(mn, mx, bits, meta_f16);
        if (lane == 0) {
            if (scale) scale[row * ng + g] = m.scale;
            if (lo) lo[row * ng + g] = m.lo;
        }
        for (int e = lane; e < group; e += WAVE) {
            const int j = g * group + e;
            if (j >= d) break;
            const int c = quant_code(xr[j], m, bits);
            if (codes) codes[row * d + j] = static_cast<uint8_t>(c);
            if (deq) deq[row * d + j] = dequant(c, m);
        }
    }
}

// The same for groups of 16 to 256 channels (a power of two) and rows of whole
// float4s: L = group / 4 lanes own a group, one float4 each, so the minimum and
// maximum meet over L lanes only, x is read once with 16-byte loads and the
// codes need no division (quant_codes). Bound by HBM: 65536 rows of 128, deq
// alone, 28.5 -> 11.5 us (2.4 -> 5.8 TB/s).
template <int L>
__global__ void __launch_bounds__(256) quantize_groups_kernel(const float* __restrict__ x, uint32_t n_groups_all, int ng,
                                                              int d, int bits, int meta_f16, uint8_t* codes,
                                                              float* scale, float* lo, float* deq) {
    const uint32_t gid = (uint32_t)blockIdx.x * (256 / L) + threadIdx.x / L;
    if (gid >= n_groups_all) return;   // whole lane groups
    const int l = threadIdx.x % L;
    const uint32_t row = gid / ng, g = gid % ng;
    const int j = g * (4 * L) + 4 * l;
    const bool in = j < d;             // past d: the zero padding of a short last group
    const int64_t at = (int64_t)row * d + j;
    const float4 u = in ? *reinterpret_cast<const float4*>(x + at) : make_float4(0.f, 0.f, 0.f, 0.f);
    const float v[4] = {u.x, u.y, u.z, u.w};
    // from the identities, as the rows kernel: a group of NaNs alone has lo = +inf there
    float mn = INFINITY, mx = -INFINITY;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        mn = fminf(mn, v[e]);
        mx = fmaxf(mx, v[e]);
    }
#pragma unroll
    for (int o = L / 2; o > 0; o >>= 1) {
        mn = fminf(mn, __shfl_xor(mn, o));
        mx = fmaxf(mx, __shfl_xor(mx, o));
    }
    const GroupMeta m = group_meta(mn, mx, bits, meta_f16);
    if (l == 0) {
        if (scale) scale[gid] = m.scale;
        if (lo) lo[gid] = m.lo;
    }
    uint32_t c[4];
    quant_codes(v, m, bits, c);
    if (!in) return;
    if (codes) *reinterpret_cast<uint32_t*>(codes + at) = c[0] | c[1] << 8 | c[2] << 16 | c[3] << 24;
    if (deq)
        *reinterpret_cast<float4*>(deq + at) = make_float4(dequant(c[0], m), dequant(c[1], m), dequant(c[2], m), dequant(c[3], m));
}

}  // namespace dkv

extern "C" int dkv_quantize(const float* x, int64_t rows, int32_t d, int32_t bits, int32_t group,
                            int32_t meta_f16, uint8_t* codes, float* scale, float* lo, float* deq,
                            dkv_stream_t stream) {
    DKV_REQUIRE(x != nullptr, "dkv_quantize: x is NULL");
    DKV_REQUIRE(rows >= 0 && d > 0, "dkv_quantize: rows must be >= 0 and d > 0");
    DKV_REQUIRE(bits == 2 || bits == 3 || bits == 4 || bits == 8, "dkv_quantize: bits must be 2, 3, 4 or 8");
    DKV_REQUIRE(group > 0, "dkv_quantize: group must be > 0");
    if (rows == 0) return DKV_OK;
    // the vector kernel's groups and rows, as far as its `all` * `lanes` threads fit a launch (2^32); the rows
    // kernel takes any, and rows wider than 256 channels further than that
    const int ng = dkv::n_groups(d, group), lanes = group / 4;
    const int64_t all = rows * ng;
    auto aligned = [](const void* p, int n) { return reinterpret_cast<uintptr_t>(p) % n == 0; };
    if (group >= 16 && group <= 256 && (group & (group - 1)) == 0 && d % 4 == 0 && all <= ((1LL << 32) - 256) / lanes && aligned(x, 16) &&
        aligned(deq, 16) && aligned(codes, 4)) {
#define DKV_QUANT(LL)                                                                                              \
    hipLaunchKernelGGL(dkv::quantize_groups_kernel<LL>, dim3((unsigned)((all + 256 / LL - 1) / (256 / LL))),       \
                       dim3(256), 0, dkv::as_stream(stream), x, (uint32_t)all, ng, d, bits, meta_f16, codes, scale, \
                       lo, deq)
        switch (lanes) {
            case 4: DKV_QUANT(4); break;
            case 8: DKV_QUANT(8); break;
            case 16: DKV_QUANT(16); break;
            case 32: DKV_QUANT(32); break;
            default: DKV_QUANT(64); break;
        }
#undef DKV_QUANT
        return dkv::check_launch("dkv_quantize");
    }
    const int waves = 4;
    const int64_t blocks = (rows + waves - 1) / waves;
    DKV_REQUIRE(blocks < (1LL << 31), "dkv_quantize: too many rows");
    hipLaunchKernelGGL(dkv::quantize_rows_kernel, dim3((unsigned)blocks), dim3(64 * waves), 0,
                       dkv::as_stream(stream), x, rows, d, bits, group, meta_f16, codes, scale, lo, deq);
    return dkv::check_launch("dkv_quantize");
}

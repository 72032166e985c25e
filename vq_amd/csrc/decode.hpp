// Reconstruction from codes: out[i][s] = centroid codes[i][s] of column block s, as binary16 or f32.
#pragma once
#include <hip/hip_fp16.h>
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace vq {

typedef uint32_t u32x4_out __attribute__((ext_vector_type(4)));

// One thread makes four 16-byte pieces of the output, 256 pieces apart, so that a wave stores 1 KB of consecutive
// bytes at a time: a centroid's eight components rounded to binary16 (F16; sd a multiple of 8) or four f32 (sd a multiple
// of 4), read from the table through the vector cache.  The workgroup's first piece is divided once, the
// others' places follow in 32 bits; the stores pass the caches (83 -> 79 us).  Bound by the stores.  1M leaves of a
// tree over 128 floats, launch and wait included: 106 us with 8 bytes per lane and a 64-bit division each
// (k_tsvq_decode4_f16), 79 so; 100,000 x 4 blocks of 32, k = 600: 25 -> 22.
template <bool F16, typename CodeT>
__global__ void __launch_bounds__(256) k_decode_gather(const CodeT *__restrict__ codes, int64_t n, int m, int sd, int k,
                                                       const float *__restrict__ cb, u32x4_out *__restrict__ out) {
    const uint32_t pieces = (uint32_t)sd / (F16 ? 8u : 4u), per_row = pieces * (uint32_t)m;
    const int64_t first = (int64_t)blockIdx.x * 1024, total = n * per_row;
    const int64_t row0 = first / per_row;  // uniform
    const uint32_t rem0 = (uint32_t)(first - row0 * per_row);
    const float4 *src[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) {
        uint32_t local = rem0 + threadIdx.x + 256u * u;
        if (first + threadIdx.x + 256 * u >= total) local = rem0;  // (not stored)
        const uint32_t dr = local / per_row, c = local - dr * per_row;
        const uint32_t s = pieces == 1 ? c : c / pieces, pc = c - s * pieces;
        const size_t code = (size_t)codes[(row0 + dr) * m + s];
        src[u] = reinterpret_cast<const float4 *>(cb + ((size_t)s * k + code) * sd) + (F16 ? 2 : 1) * pc;
    }
    float4 a[4], b[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) {
        a[u] = src[u][0];
        b[u] = F16 ? src[u][1] : a[u];
    }
#pragma unroll
    for (int u = 0; u < 4; ++u) {
        u32x4_out v;
        if constexpr (F16) {
            auto two = [](float lo, float hi) {  // round to nearest even
                return (uint32_t)__half_as_ushort(__float2half_rn(lo)) | ((uint32_t)__half_as_ushort(__float2half_rn(hi)) << 16);
            };
            v = u32x4_out{two(a[u].x, a[u].y), two(a[u].z, a[u].w), two(b[u].x, b[u].y), two(b[u].z, b[u].w)};
        } else {
            v = u32x4_out{__float_as_uint(a[u].x), __float_as_uint(a[u].y), __float_as_uint(a[u].z), __float_as_uint(a[u].w)};
        }
        const int64_t at = first + threadIdx.x + 256 * u;
        if (at < total) __builtin_nontemporal_store(v, out + at);
    }
}

}  // namespace vq

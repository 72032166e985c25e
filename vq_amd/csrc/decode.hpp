// Reconstruction from codes: out[i][s] = centroid codes[i][s] of column block s, as binary16 or f32 (the leaves of a tree,
// src/tsvq.rs:242-248: one block whose entries are the nodes).
#pragma once
#include <hip/hip_fp16.h>
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <type_traits>

#include "resident_rules.hpp"

namespace vq {

typedef uint32_t u32x4_out __attribute__((ext_vector_type(4)));

// One thread makes four 16-byte pieces of the output, 256 pieces apart, so that a wave stores 1 KB of consecutive
// bytes at a time: a centroid's eight components rounded to binary16 (F16; sd a multiple of 8) or four f32 (sd a multiple
// of 4), read from the table through the vector cache.  The workgroup's first piece is divided once, the
// others' places follow in 32 bits; the stores pass the caches (83 -> 79 us).  Bound by the stores.  1M leaves of a
// tree over 128 floats, launch and wait included: 106 us with 8 bytes per lane and a 64-bit division each,
// 79 so; 100,000 x 4 blocks of 32, k = 600: 25 -> 22.
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

// The same for blocks of any width and outputs of any alignment, UNIT consecutive components (1, 2 or 4, a divisor of the
// width) per read of the table and store; U of them in flight per thread, 256 apart.  Places are counted from the workgroup's first
// block on and divided in 32 bits: a thread per component with two divisions in 64 bits wrote 0.9-1.0 TB/s at any size (372,160 x 21
// blocks of 15 229 us, 147 so; 181,650 x 33 of 6 77 -> 32; f16 blocks of 4 as before, 1.7-2.1 TB/s).  Bound by the vector
// caches' gather of the codes and the table, which decode_flat_resident's sizes have in LDS.
template <bool F16, int UNIT, int U, typename CodeT>
__global__ void __launch_bounds__(256) k_decode_units(const CodeT *__restrict__ codes, int64_t n, int m, int sd, int k,
                                                      const float *__restrict__ cb, void *__restrict__ outv) {
    using OutT = typename std::conditional<F16, uint16_t, float>::type;
    constexpr int RUN = 256 * U * UNIT;
    const int64_t blocks = n * m, total = blocks * sd, first = (int64_t)blockIdx.x * RUN;
    const float *src[U];
    if (m == 1 && total <= 0xFFFFFFFFll) {  // the rows of a tree: one division on the way to the code (20,000 x 100 with its descent 25.4 -> 24.8 us)
#pragma unroll
        for (int u = 0; u < U; ++u) {
            uint32_t e = (uint32_t)first + (threadIdx.x + 256u * u) * UNIT;
            if (first + (threadIdx.x + 256u * u) * UNIT >= total) e = (uint32_t)first;  // (not stored)
            const uint32_t b = e / (uint32_t)sd;
            src[u] = cb + (size_t)codes[b] * sd + (e - b * (uint32_t)sd);
        }
    } else {
        const int64_t b0 = total <= 0xFFFFFFFFll ? (uint32_t)first / (uint32_t)sd : first / sd;  // uniform
        const uint32_t t0 = (uint32_t)(first - b0 * sd), s0 = total <= 0xFFFFFFFFll ? (uint32_t)b0 % (uint32_t)m : (uint32_t)(b0 % m);
        const CodeT *run = codes + b0;
#pragma unroll
        for (int u = 0; u < U; ++u) {
            uint32_t e = t0 + (threadIdx.x + 256u * u) * UNIT;
            if (first + (threadIdx.x + 256u * u) * UNIT >= total) e = t0;  // (not stored)
            const uint32_t b = e / (uint32_t)sd, t = e - b * (uint32_t)sd, s = s0 + b;
            src[u] = cb + ((size_t)(s - s / (uint32_t)m * (uint32_t)m) * k + (size_t)run[b]) * sd + t;
        }
    }
    typedef float fv __attribute__((ext_vector_type(UNIT == 1 ? 2 : UNIT)));  // (of two, one is used where UNIT is 1)
    fv v[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
        if constexpr (UNIT == 1) v[u][0] = *src[u];
        else v[u] = *reinterpret_cast<const fv *>(src[u]);
    }
    const bool whole = (reinterpret_cast<uintptr_t>(outv) & (UNIT * sizeof(OutT) - 1)) == 0;  // uniform
#pragma unroll
    for (int u = 0; u < U; ++u) {
        const int64_t at = first + (threadIdx.x + 256u * u) * UNIT;
        if (at >= total) continue;
        OutT *out = reinterpret_cast<OutT *>(outv) + at;
        typedef OutT ov __attribute__((ext_vector_type(UNIT == 1 ? 2 : UNIT)));
        ov o;
#pragma unroll
        for (int i = 0; i < UNIT; ++i) {
            if constexpr (F16) o[i] = __half_as_ushort(__float2half_rn(v[u][i]));
            else o[i] = v[u][i];
        }
        if (UNIT > 1 && whole) {
            *reinterpret_cast<ov *>(out) = o;
        } else {
#pragma unroll
            for (int i = 0; i < UNIT; ++i) out[i] = o[i];
        }
    }
}

// f16 rows (16-byte aligned) of blocks of any width with the table of all blocks in LDS (up to 160 KB; one workgroup of 1024 threads per compute
// unit, two up to 80 KB): a thread makes eight consecutive components per step whatever blocks they belong to, two steps in flight,
// so a wave stores 1 KB of consecutive bytes.  FEW: eight components lie in two blocks at most, whose codes are read once.
// The stores (4.0 TB/s at 372,160 x 315) or, in narrow blocks, the LDS reads and the codes bound it.
template <int UNIT, bool FEW, typename CodeT>
__global__ void __launch_bounds__(1024) k_decode_flat(const CodeT *__restrict__ codes, int64_t n, int m, int sd, int k,
                                                      const float *__restrict__ cb, uint16_t *__restrict__ out) {
    constexpr int PER = 8, STEPS = 2, T = 1024, RUN = T * STEPS * PER;
    extern __shared__ __attribute__((aligned(16))) uint16_t flat_tab[];  // [m * k][sd]
    const uint32_t entries = (uint32_t)m * k * sd;
    auto two = [](float lo, float hi) {
        return (uint32_t)__half_as_ushort(__float2half_rn(lo)) | ((uint32_t)__half_as_ushort(__float2half_rn(hi)) << 16);
    };
    const uint32_t quads = (reinterpret_cast<uintptr_t>(cb) & 15) == 0 ? entries / 4 : 0;
#pragma unroll 4
    for (uint32_t e = threadIdx.x; e < quads; e += T) {
        const float4 v = reinterpret_cast<const float4 *>(cb)[e];
        reinterpret_cast<uint2 *>(flat_tab)[e] = make_uint2(two(v.x, v.y), two(v.z, v.w));
    }
    for (uint32_t e = 4 * quads + threadIdx.x; e < entries; e += T) flat_tab[e] = (uint16_t)two(cb[e], 0.0f);
    __syncthreads();
    const int64_t blocks = n * m, total = blocks * sd;
    for (int64_t first = (int64_t)blockIdx.x * RUN; first < total; first += (int64_t)gridDim.x * RUN) {
        const int64_t b0 = total <= 0xFFFFFFFFll ? (uint32_t)first / (uint32_t)sd : first / sd;  // uniform
        const uint32_t t0 = (uint32_t)(first - b0 * sd), s0 = total <= 0xFFFFFFFFll ? (uint32_t)b0 % (uint32_t)m : (uint32_t)(b0 % m);
        const CodeT *run = codes + b0;
        const uint32_t last = blocks - 1 - b0 < RUN ? (uint32_t)(blocks - 1 - b0) : (uint32_t)RUN;  // no block is read beyond it
#pragma unroll
        for (int u = 0; u < STEPS; ++u) {
            const uint32_t off = (threadIdx.x + T * u) * PER, e = t0 + off;
            uint32_t b = e / (uint32_t)sd, t = e - b * (uint32_t)sd, s = s0 + b, code = 0, next = 0;
            s -= s / (uint32_t)m * (uint32_t)m;
            if constexpr (FEW) {
                code = (uint32_t)run[b < last ? b : last];
                next = (uint32_t)run[b + 1 < last ? b + 1 : last];
            }
            uint32_t w[PER / 2];  // pairs of components
#pragma unroll
            for (int i = 0; i < PER; i += UNIT) {
                if constexpr (!FEW) code = (uint32_t)run[b < last ? b : last];
                const uint16_t *p = flat_tab + ((s * (uint32_t)k + code) * (uint32_t)sd + t);
                if constexpr (UNIT == 1) {
                    if (i % 2 == 0) w[i / 2] = *p;
                    else w[i / 2] |= (uint32_t)*p << 16;
                } else if constexpr (UNIT == 2) {
                    w[i / 2] = *reinterpret_cast<const uint32_t *>(p);
                } else {
                    const uint2 x = *reinterpret_cast<const uint2 *>(p);
                    w[i / 2] = x.x, w[i / 2 + 1] = x.y;
                }
                t += UNIT;
                if (t == (uint32_t)sd) {
                    t = 0;
                    ++b;
                    s = s + 1 == (uint32_t)m ? 0u : s + 1;
                    if constexpr (FEW) code = next;
                }
            }
            const int64_t left = total - first - off;
            if (left >= PER) {
                __builtin_nontemporal_store(u32x4_out{w[0], w[1], w[2], w[3]}, reinterpret_cast<u32x4_out *>(out + first + off));
            } else {
#pragma unroll
                for (int i = 0; i < PER; ++i)
                    if (i < left) out[first + off + i] = (uint16_t)(w[i / 2] >> (16 * (i % 2)));
            }
        }
    }
}

// Widths and alignments that k_decode_gather does not take, launched.  k: entries per block (of a tree: its nodes).
// lds_set: the caller's, a bit per kernel whose LDS limit has been set.  The table only for aligned outputs: with single stores of the
// others 500,000 blocks of 5 take 3.1 us more than aligned ones, from memory 1.2 (200,000 x 10 of 10 42 us against 32 from memory).  Four
// units in flight per thread against one: 20,000 x 20 of 9 19.1 us against 20.8, 20,000 x 40 of 10 20.6 against 22.8; of 12, whose units are four
// components, 20,000 rows 20.7 against 20.1, 25,000 21.9 against 21.4, 1,000,000 x 4 of 4 23.5 against 24.3.
template <bool F16, typename CodeT>
hipError_t launch_decode_any(hipStream_t st, int compute_units, uint32_t &lds_set, const CodeT *codes, int64_t n, int m, int sd, int k,
                             const float *cb, void *out) {
    const bool whole = (reinterpret_cast<uintptr_t>(out) & 15) == 0;
    const size_t lds = F16 && whole && decode_flat_resident(n, m, sd, k) ? 2 * (size_t)m * k * sd : 0;
    const unsigned lds_groups = (unsigned)compute_units * (lds <= kDecodeFlatLds / 2 ? 2u : 1u);
    const uintptr_t at = reinterpret_cast<uintptr_t>(cb);
    const int64_t total = n * m * sd;
    auto go = [&](auto U) -> hipError_t {
        constexpr int UNIT = decltype(U)::value;
        if constexpr (F16) {
            if (lds) {
                auto kern = sd >= 8 - UNIT ? k_decode_flat<UNIT, true, CodeT> : k_decode_flat<UNIT, false, CodeT>;
                const uint32_t bit = 1u << ((UNIT / 2 * 2 + (sd >= 8 - UNIT ? 1 : 0)) * 3 + sizeof(CodeT) / 2);
                if (!(lds_set & bit)) {
                    const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void *>(kern),
                                                             hipFuncAttributeMaxDynamicSharedMemorySize, kDecodeFlatLds);
                    if (e != hipSuccess) return e;
                    lds_set |= bit;
                }
                const int64_t runs = (total + 16383) / 16384;
                hipLaunchKernelGGL(kern, dim3((unsigned)(runs < lds_groups ? runs : lds_groups)), dim3(1024), lds, st, codes, n, m, sd, k,
                                   cb, (uint16_t *)out);
                return hipSuccess;
            }
        }
        const bool one = total < (UNIT == 4 ? 3 << 22 : UNIT << 21);
        auto kern = one ? k_decode_units<F16, UNIT, 1, CodeT> : k_decode_units<F16, UNIT, 4, CodeT>;
        const int64_t run = (one ? 256 : 1024) * UNIT;
        hipLaunchKernelGGL(kern, dim3((unsigned)((total + run - 1) / run)), dim3(256), 0, st, codes, n, m, sd, k, cb, out);
        return hipSuccess;
    };
    if (sd % 4 == 0 && at % 16 == 0) return go(std::integral_constant<int, 4>{});
    return sd % 2 == 0 && at % 8 == 0 ? go(std::integral_constant<int, 2>{}) : go(std::integral_constant<int, 1>{});
}

}  // namespace vq

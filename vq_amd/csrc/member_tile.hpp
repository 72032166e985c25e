// Sums over the members of a list in list order: what the leaf sums of a fit, the means of a cluster and the variances of
// a tree node have in common.
//
// This translation unit must be compiled with -ffp-contract=off.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace vq {

// The sum of members lo .. hi - 1 of a list (row_of: position -> row) over a tile of up to VEC P components, by a
// workgroup: P pieces of VEC floats per member; the threads fetch a chunk of members into registers, eight loads of each in
// flight while the chunk before is added, and store them transposed in LDS (stage: width * (8 NT / P + 4) floats); a lane per
// component adds them in list order, sixteen members read at a time (with the next sixteen read
// beside the adds no faster).  xs: row 0's tile.  Returned in the lanes
// below width.  The last piece of a tile begins at the tile's end less VEC, so that pieces of any width are whole (what
// two of them share is written twice, with the same values).  Its time is a chain of memory round trips, one per chunk of 128
// to 512 members, beside the adds: 7,930 x 300, k = 22 41 -> 17 us per launch, 50,019 x 28 blocks of 10, k = 78 110 -> 28.
// (With chunks of twice the members by 256 threads the same, where the leaves are long; the LDS then holds half the leaves.)
// DEV: of the squared deviations from mean (the tile's), two roundings each, made as they are stored.
template <int NT, int VEC, bool DEV = false, typename RowOf>
__device__ __forceinline__ float member_tile_sum(float *stage, const float *__restrict__ xs, int64_t ld, uint32_t lo, uint32_t hi, int width,
                                                 int pieces, RowOf row_of, const float *__restrict__ mean = nullptr) {
    typedef float piece_t __attribute__((ext_vector_type(VEC), aligned(4)));
    constexpr int E = 8;
    const int tid = threadIdx.x;
    const int step = NT / pieces, mine = tid / pieces, at = VEC * (tid % pieces);
    const int t0 = at + VEC <= width ? at : width - VEC;
    const bool fetches = mine < step;
    xs += t0;
    const uint32_t chunk = (uint32_t)(E * step), stride = chunk + 4;
    uint32_t row[E];
    piece_t v[E], mu;
    if constexpr (DEV) mu = *reinterpret_cast<const piece_t *>(mean + t0);
    auto rows = [&](uint32_t p) {  // past the end: the last member's
#pragma unroll
        for (int i = 0; i < E; ++i) {
            const uint32_t q = p + (uint32_t)(mine + step * i);
            row[i] = row_of(q < hi ? q : hi - 1);
        }
    };
    auto load = [&](uint32_t p) {
#pragma unroll
        for (int i = 0; i < E; ++i)
            if (p + (uint32_t)(step * i) < hi) v[i] = *reinterpret_cast<const piece_t *>(xs + (int64_t)row[i] * ld);
    };
    float acc = 0.0f;
    if (fetches && lo < hi) {
        rows(lo);
        load(lo);
    }
    for (uint32_t p = lo; p < hi; p += chunk) {
        const uint32_t cm = hi - p < chunk ? hi - p : chunk;
        if (fetches && p + chunk < hi) rows(p + chunk);
        if (p != lo) __syncthreads();  // the chunk before has been added
        if (fetches) {
#pragma unroll
            for (int i = 0; i < E; ++i)
                if ((uint32_t)(step * i) < cm)
#pragma unroll
                    for (int e = 0; e < VEC; ++e) {
                        float put = v[i][e];
                        if constexpr (DEV) {
                            const float d = put - mu[e];
                            put = d * d;
                        }
                        stage[(uint32_t)(t0 + e) * stride + (uint32_t)(mine + step * i)] = put;
                    }
            if (p + chunk < hi) load(p + chunk);
        }
        __syncthreads();
        if (tid < width) {
            const float *col = stage + (uint32_t)tid * stride;
            uint32_t mbr = 0;
            for (; mbr + 16 <= cm; mbr += 16) {
                float4 q[4];
#pragma unroll
                for (int u = 0; u < 4; ++u) q[u] = *reinterpret_cast<const float4 *>(col + mbr + 4 * u);
#pragma unroll
                for (int u = 0; u < 4; ++u) {
                    acc = acc + q[u].x;
                    acc = acc + q[u].y;
                    acc = acc + q[u].z;
                    acc = acc + q[u].w;
                }
            }
            for (; mbr < cm; ++mbr) acc = acc + col[mbr];
        }
    }
    return acc;
}

}  // namespace vq

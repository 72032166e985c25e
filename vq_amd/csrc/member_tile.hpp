// Sums over the members of a list in list order: what the leaf sums of a fit, the means of a cluster and the variances of
// a tree node have in common.
//
// This translation unit must be compiled with -ffp-contract=off.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace vq {

// acc and the count values of a column in LDS (16-byte aligned), one after the other: sixteen are added while the next sixteen are
// read.  The scheduler is held to that order: left to itself it puts the reads behind the adds, and every sixteen members
// wait for LDS.  (A chain alone on its compute unit gains by it; where other workgroups fill the wait the registers cost more:
// add_column_plain.)
__device__ __forceinline__ float add_column(const float *col, uint32_t count, float acc) {
    float4 q[2][4];
    auto read = [&](float4 (&d)[4], uint32_t at) {
#pragma unroll
        for (int u = 0; u < 4; ++u) d[u] = *reinterpret_cast<const float4 *>(col + at + 4 * u);
        __builtin_amdgcn_sched_barrier(0);
    };
    auto add = [&](const float4 (&d)[4]) {
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            acc = acc + d[u].x;
            acc = acc + d[u].y;
            acc = acc + d[u].z;
            acc = acc + d[u].w;
        }
        __builtin_amdgcn_sched_barrier(0);
    };
    uint32_t m = 0;
    if (count >= 16) {
        read(q[0], 0);
        for (; m + 48 <= count; m += 32) {
            read(q[1], m + 16);
            add(q[0]);
            read(q[0], m + 32);
            add(q[1]);
        }
        if (m + 32 <= count) {
            read(q[1], m + 16);
            add(q[0]);
            add(q[1]);
            m += 32;
        } else {
            add(q[0]);
            m += 16;
        }
    }
    for (; m < count; ++m) acc = acc + col[m];
    return acc;
}

// The same, sixteen read and then added.
__device__ __forceinline__ float add_column_plain(const float *col, uint32_t count, float acc) {
    uint32_t m = 0;
    for (; m + 16 <= count; m += 16) {
        float4 q[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) q[u] = *reinterpret_cast<const float4 *>(col + m + 4 * u);
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            acc = acc + q[u].x;
            acc = acc + q[u].y;
            acc = acc + q[u].z;
            acc = acc + q[u].w;
        }
    }
    for (; m < count; ++m) acc = acc + col[m];
    return acc;
}

// The sum of members lo .. hi - 1 of a list (row_of: position -> row) over a tile of up to VEC P components, by a
// workgroup: P pieces of VEC floats per member; the threads fetch a chunk of members into registers, eight loads of each in
// flight while the chunk before is added, and store them transposed in LDS (stage: width * (8 NT / P + 4) floats); a lane per
// component adds them in list order, sixteen members read at a time.  xs: row 0's tile.  Returned in the lanes
// below width.  The last piece of a tile begins at the tile's end less VEC, so that pieces of any width are whole (what
// two of them share is written twice, with the same values).  Its time is a chain of memory round trips, one per chunk of 128
// to 512 members, beside the adds (reading ahead as add_column does costs fits 1 to 3 %: 84,443 x 100, k = 108 3351 -> 3424 us): 7,930 x 300, k = 22 41 -> 17 us per launch, 50,019 x 28 blocks of 10, k = 78 110 -> 28.
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
        if (tid < width) acc = add_column_plain(stage + (uint32_t)tid * stride, cm, acc);
    }
    return acc;
}

// The same where a chain of adds decides (few workgroups, long lists): the first wave adds, the others fetch, and two
// stages take turns, so that a chunk's way into LDS lies beside the adds of the one before and a chunk costs one barrier.
// stage: 2 * width * (kChainE (NT - 64) / P + 4) floats.  NT: 128 or more.
constexpr int kChainE = 7;
__host__ __device__ constexpr size_t chain_stage_floats(int nt, int width, int pieces) {
    return 2 * (size_t)width * (size_t)(kChainE * ((nt - 64) / pieces) + 4);
}
template <int NT, int VEC, bool DEV = false, typename RowOf>
__device__ __forceinline__ float member_chain_sum(float *stage, const float *__restrict__ xs, int64_t ld, uint32_t lo, uint32_t hi, int width,
                                                  int pieces, RowOf row_of, const float *__restrict__ mean = nullptr) {
    typedef float piece_t __attribute__((ext_vector_type(VEC), aligned(4)));
    constexpr int E = kChainE;
    const int tid = threadIdx.x, ft = tid - 64;  // (the first wave adds)
    const int step = (NT - 64) / pieces, mine = ft / pieces, at = VEC * (ft % pieces);
    const int t0 = at + VEC <= width ? at : width - VEC;
    const bool fetches = ft >= 0 && mine < step;
    const uint32_t chunk = (uint32_t)(E * step), stride = chunk + 4, size = (uint32_t)width * stride;
    uint32_t row[E];
    piece_t v[E], mu;
    if constexpr (DEV)
        if (fetches) mu = *reinterpret_cast<const piece_t *>(mean + t0);
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
            if (p + (uint32_t)(step * i) < hi) v[i] = *reinterpret_cast<const piece_t *>(xs + t0 + (int64_t)row[i] * ld);
    };
    auto put = [&](uint32_t p, float *to) {
#pragma unroll
        for (int i = 0; i < E; ++i)
            if (p + (uint32_t)(step * i) < hi)
#pragma unroll
                for (int e = 0; e < VEC; ++e) {
                    float w = v[i][e];
                    if constexpr (DEV) {
                        const float d = w - mu[e];
                        w = d * d;
                    }
                    to[(uint32_t)(t0 + e) * stride + (uint32_t)(mine + step * i)] = w;
                }
    };
    float acc = 0.0f;
    if (fetches && lo < hi) {
        rows(lo);
        load(lo);
        if (lo + chunk < hi) rows(lo + chunk);
        put(lo, stage);
        if (lo + chunk < hi) load(lo + chunk);
    }
    uint32_t buf = 0;
    for (uint32_t p = lo; p < hi; p += chunk, buf ^= 1) {
        __syncthreads();  // this chunk is in its stage, and the other stage has been added
        if (fetches) {
            if (p + chunk < hi) {
                if (p + 2 * chunk < hi) rows(p + 2 * chunk);
                put(p + chunk, stage + (buf ^ 1) * size);
                if (p + 2 * chunk < hi) load(p + 2 * chunk);
            }
        } else if (tid < width) {
            acc = add_column(stage + buf * size + (uint32_t)tid * stride, hi - p < chunk ? hi - p : chunk, acc);
        }
    }
    return acc;
}

// One or the other.  Chains are the faster ones while the workgroups, at 44 KB of LDS for 16 components, are a round of the GPU
// (kChainGroups on a compute unit); beyond, more fetching threads in each are.  100,000 x 128, the levels of 16, 32 and 64 nodes 28.5 -> 20.6 us on average, of 128 and 256 nodes (1024 and 2048 workgroups) 22.7 -> 28.0;
// 4,157 x 100, of one, two and four nodes 20.2 -> 15.2.
constexpr int kChainGroups = 3;
template <int NT, int VEC, bool DEV, bool CHAIN, typename RowOf>
__device__ __forceinline__ float tile_sum(float *stage, const float *__restrict__ xs, int64_t ld, uint32_t lo, uint32_t hi, int width, int pieces,
                                          RowOf row_of, const float *__restrict__ mean = nullptr) {
    if constexpr (CHAIN) return member_chain_sum<NT, VEC, DEV>(stage, xs, ld, lo, hi, width, pieces, row_of, mean);
    else return member_tile_sum<NT, VEC, DEV>(stage, xs, ld, lo, hi, width, pieces, row_of, mean);
}

}  // namespace vq

// Tree-structured VQ: node statistics for the build (src/tsvq.rs:71-148) and the descent
// encode (src/tsvq.rs:162-181).
//
// Build, one tree level at a time.  `perm` lists row ids so that the rows of every node of the
// level are contiguous and in original row order (the reference's partition is stable).
//   mean      mean_vector over the node's rows: sequential up to 1024 rows, the fixed midpoint
//             tree above (same order as the LBG update)
//   variance  per dimension, sum over the node's rows IN ROW ORDER of (x - mean)^2, f32
//             (Iterator::sum is sequential, src/tsvq.rs:88-99) — one lane per (node, dimension)
//   median    of the split column by a segmented sort (host picks the middle values)
//   partition stable, by `x[split] <= median`
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "assign_exact.hpp"
#include "member_tile.hpp"

namespace vq {

// One lane per (leaf, component): sequential sum over perm[lo, hi).
static __global__ void __launch_bounds__(256) k_seg_leafsum(const uint32_t *__restrict__ perm,
                                                     const uint2 *__restrict__ desc, int64_t nleaves,
                                                     const float *__restrict__ x, int64_t ld, int sd,
                                                     float *__restrict__ leaf_sum) {
    int64_t gid = (int64_t)blockIdx.x * 256 + threadIdx.x;
    int64_t leaf = gid / sd;
    int t = (int)(gid % sd);
    if (leaf >= nleaves) return;
    uint2 d = desc[leaf];
    const float *__restrict__ xc = x + t;
    float acc = 0.0f;
    // a leaf has up to 1024 rows and the lane adds them one after the other: 32 loads are in
    // flight per memory round trip (unconditional, clamped to the leaf's last row), the adds keep
    // their order
    uint32_t p = d.x;
    if (d.y > d.x) {
        const uint32_t last = d.y - 1;
        for (; p < d.y; p += 32) {
            uint32_t id[32];
            float v[32];
#pragma unroll
            for (int u = 0; u < 32; ++u) id[u] = perm[p + u <= last ? p + u : last];
#pragma unroll
            for (int u = 0; u < 32; ++u) v[u] = xc[(int64_t)id[u] * ld];
#pragma unroll
            for (int u = 0; u < 32; ++u)
                if (p + u <= last) acc = acc + v[u];
        }
    }
    leaf_sum[leaf * sd + t] = acc;
}

// The same sums where there are too few of them to fill the chip with a lane each: a workgroup takes 32
// components of a leaf, all of its threads bring the rows in, 128 at a time through LDS, and one half wave
// adds them in order while the next tile is on its way (the row numbers a tile ahead of the rows).
// 128 leaves of 782 rows of 128 (100,000 rows): 31 -> 13 us, a level of the tree each.
static __global__ void __launch_bounds__(256) k_seg_leafsum_wg(const uint32_t *__restrict__ perm,
                                                               const uint2 *__restrict__ desc,
                                                               const float *__restrict__ x, int64_t ld, int sd,
                                                               float *__restrict__ leaf_sum) {
    __shared__ float tile[2][128][32];
    const int64_t leaf = blockIdx.x;
    const int c = threadIdx.x & 31, sub = threadIdx.x >> 5, t = blockIdx.y * 32 + c;
    const uint2 d = desc[leaf];
    const float *xc = x + (t < sd ? t : 0);
    float acc = 0.0f;
    if (d.y > d.x) {
        const uint32_t last = d.y - 1;
        uint32_t id[16];
        float v[16];
        auto ids = [&](uint32_t p) {
#pragma unroll
            for (int u = 0; u < 16; ++u) id[u] = perm[p + 8 * u + sub <= last ? p + 8 * u + sub : last];
        };
        auto rows = [&]() {
#pragma unroll
            for (int u = 0; u < 16; ++u) v[u] = xc[(int64_t)id[u] * ld];
        };
        ids(d.x);
        rows();
        ids(d.x + 128);
        int buf = 0;
        for (uint32_t p = d.x; p < d.y; p += 128, buf ^= 1) {
#pragma unroll
            for (int u = 0; u < 16; ++u) tile[buf][8 * u + sub][c] = v[u];
            rows();  // (past the leaf: its last row again, not added)
            ids(p + 256);
            __syncthreads();
            if (threadIdx.x < 32) {
                const uint32_t left = d.y - p;
                if (left >= 128) {
#pragma unroll 32
                    for (int r = 0; r < 128; ++r) acc = acc + tile[buf][r][c];
                } else {
#pragma unroll 8
                    for (uint32_t r = 0; r < left; ++r) acc = acc + tile[buf][r][c];
                }
            }
        }
    }
    if (threadIdx.x < 32 && t < sd) leaf_sum[leaf * sd + t] = acc;
}

// One lane per (segment, component): combine 2^depth leaves left + right, divide by the count.
// seg_info[g] = {first leaf, depth, count, unused}
static __global__ void __launch_bounds__(256) k_seg_mean(float *__restrict__ leaf_sum,
                                                  const uint4 *__restrict__ seg_info, int nseg, int sd,
                                                  float *__restrict__ out, int64_t out_first) {
    int64_t gid = (int64_t)blockIdx.x * 256 + threadIdx.x;
    int g = (int)(gid / sd);
    int t = (int)(gid % sd);
    if (g >= nseg) return;
    uint4 info = seg_info[g];
    uint32_t nl = 1u << info.y;
    float *ls = leaf_sum + (size_t)info.x * sd + t;
    // the pairs of one level of the tree are independent: eight of them per memory round trip
    // (clamped to the level's last pair); a lane only reads what it wrote itself
    for (uint32_t h = 1; h < nl; h <<= 1) {
        const uint32_t npairs = nl / (2 * h);
        for (uint32_t q0 = 0; q0 < npairs; q0 += 8) {
            float a[8], b[8];
#pragma unroll
            for (uint32_t u = 0; u < 8; ++u) {
                const uint32_t qi = q0 + u < npairs ? q0 + u : npairs - 1;
                a[u] = ls[(size_t)(2 * h * qi) * sd];
                b[u] = ls[(size_t)(2 * h * qi + h) * sd];
            }
#pragma unroll
            for (uint32_t u = 0; u < 8; ++u)
                if (q0 + u < npairs) ls[(size_t)(2 * h * (q0 + u)) * sd] = a[u] + b[u];
        }
    }
    out[(out_first + g) * sd + t] = ls[0] / __uint2float_rn(info.z);
}

// The same tree for the levels near the root, where a segment has hundreds of leaves and there are
// few segments: one workgroup per (segment, 8 components), the leaf sums in LDS, the pairs of a tree
// level side by side — the same additions as k_seg_mean, which walks them in one thread.
constexpr int kMeanWgLeaves = 1024;
static __global__ void __launch_bounds__(256) k_seg_mean_wg(const float *__restrict__ leaf_sum,
                                                            const uint4 *__restrict__ seg_info, int sd,
                                                            float *__restrict__ out, int64_t out_first) {
    __shared__ float tree[kMeanWgLeaves][8];
    const int g = blockIdx.x, t = threadIdx.x & 7, q = threadIdx.x >> 3;
    const int c = blockIdx.y * 8 + t;
    const uint4 info = seg_info[g];
    const uint32_t nl = 1u << info.y;  // <= kMeanWgLeaves (the host checks)
    const float *ls = leaf_sum + (size_t)info.x * sd + (c < sd ? c : 0);
    for (uint32_t leaf = q; leaf < nl; leaf += 32) tree[leaf][t] = ls[(size_t)leaf * sd];
    __syncthreads();
    for (uint32_t h = 1; h < nl; h <<= 1) {
        const uint32_t npairs = nl / (2 * h);
        for (uint32_t qi = q; qi < npairs; qi += 32) tree[2 * h * qi][t] = tree[2 * h * qi][t] + tree[2 * h * qi + h][t];
        __syncthreads();
    }
    if (q == 0 && c < sd) out[(out_first + g) * sd + c] = tree[0][t] / __uint2float_rn(info.z);
}

// Sums of squared deviations in row order, a workgroup per segment and tile of up to 32 components (block
// tile * nseg + segment, as y would end at 65,535 tiles; the last tile begins at dim less its width): seg_range[g] = {lo, hi} positions in perm; mean of segment g at means[(first + g) * dim].
// A chunk of 512 rows was a memory round trip, two barriers and their adds, 3.5 us in all or 7 ns a row; 4 ns where the chunks overlap the adds (CHAIN).  Against one workgroup per segment with all
// columns, whose one lane per column read its squares one by one: a root of 5,964 x 100 90 -> 41 us.
// CHAIN: few workgroups, whose chains of adds decide (member_chain_sum).
template <int VEC, bool CHAIN>
static __global__ void __launch_bounds__(256) k_seg_variance_tile(const uint32_t *__restrict__ perm, const uint2 *__restrict__ seg_range, int nseg,
                                                                 const float *__restrict__ means, int64_t first,
                                                                 const float *__restrict__ x, int64_t ld, int dim, int width, int pieces,
                                                                 float *__restrict__ var) {
    extern __shared__ float4 lds_var[];
    const int g = blockIdx.x % (unsigned)nseg, tile = blockIdx.x / (unsigned)nseg;
    const int c0 = tile * width < dim - width ? tile * width : dim - width;
    const uint2 r = seg_range[g];
    const float sum = tile_sum<256, VEC, true, CHAIN>(reinterpret_cast<float *>(lds_var), x + c0, ld, r.x, r.y, width, pieces,
                                                      [&](uint32_t p) { return perm[p]; }, means + (first + g) * dim + c0);
    if ((int)threadIdx.x < width) var[(size_t)g * dim + c0 + threadIdx.x] = sum;
}

// ---- per-dimension sums of squared deviations in two steps (dim a multiple of 8) --------------
// Step 1, on the whole GPU: sq = (x - mean)^2, the same two roundings as in the chain, stored so
// that 32 consecutive positions of a column sit side by side:
//   sq32[(lo_g + 32 g) * dim + ((p - lo_g) / 32) * 32 * dim + (c / 8) * 256 + (c % 8) * 32 + (p - lo_g) % 32]
// (every segment starts on its own group of 32 positions: n + 32 nseg rows of room).
// Grid (blocks of 64 positions, segments); one lane per (group of 32 positions, column).
constexpr int kChainGroup = 32;  // positions per group

// Index of a segment's first group in the per-group tables (group sums, binade guesses, maps):
// segment g's squares start at row range.x + 32 g of sq32, and the groups of different segments
// never share an index.
__device__ __forceinline__ size_t seg_group0(const uint2 range, int g) {
    return ((size_t)range.x + 32u * (size_t)g) / 32u;
}

static __global__ void __launch_bounds__(256) k_seg_sqdev32(const uint32_t *__restrict__ perm,
                                                            const uint2 *__restrict__ seg_range,
                                                            const float *__restrict__ means, int64_t first,
                                                            const float *__restrict__ x, int64_t ld, int dim,
                                                            float *__restrict__ sq32, float *__restrict__ gsum) {
    // sq32 == nullptr: only the group sums are wanted (the squares are made again where they are used)
    const int g = blockIdx.y;
    const uint2 range = seg_range[g];
    const uint32_t count = range.y - range.x;
    const uint32_t P0 = blockIdx.x * 2u;  // first group of this block
    if (P0 * 32u >= count) return;
    const uint32_t nP = (count + 31u) / 32u;
    const uint32_t groups = nP - P0 < 2u ? nP - P0 : 2u;
    const float *mrow = means + (first + g) * dim;
    float *out = sq32 + ((size_t)range.x + 32u * (size_t)g) * dim;
    const uint32_t *pm = perm + range.x;
    for (uint32_t e = threadIdx.x; e < groups * (uint32_t)dim; e += 256) {
        const uint32_t P = P0 + e / (uint32_t)dim, c = e % (uint32_t)dim;
        const float m = mrow[c];
        float4 *o = reinterpret_cast<float4 *>(out + (size_t)P * 32 * dim + (c / 8u) * 256u + (c % 8u) * 32u);
        float gs = 0.0f;  // the group's sum, any order: only used to guess the running sum's binade
#pragma unroll
        for (int h = 0; h < 2; ++h) {  // sixteen loads in flight at a time
            float q[16];
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                const uint32_t p = 32u * P + 16u * h + r;  // past the end: the last row again, never added
                const float d = x[(int64_t)pm[p < count ? p : count - 1] * ld + c] - m;
                q[r] = d * d;
                gs += p < count ? q[r] : 0.0f;
            }
            if (sq32)
#pragma unroll
                for (int r = 0; r < 4; ++r) o[4 * h + r] = make_float4(q[4 * r], q[4 * r + 1], q[4 * r + 2], q[4 * r + 3]);
        }
        if (gsum) gsum[(seg_group0(range, g) + P) * dim + c] = gs;
    }
}

// Step 2: the sequential sums.  Grid (segments, dim / 32); a wave owns 8 columns, eight
// neighbouring lanes own one column: lane 8 cc + j loads positions 4j .. 4j+3 of column cc of a
// group — one 16-byte load per lane moves 32 positions of 8 columns, 1 KB contiguous per wave —
// and the first lane of the eight adds the 32 values in position order, its neighbours' values
// fetched by DPP row-shift moves.  A lane keeps kChainRing loads in flight: 768
// positions per wave cover a memory round trip of 3 us at 3-4 ns per position with a ring of 96
// registers; one 16-byte load per 4 positions of a lane's own column could keep 240 in flight at
// most (the counter of outstanding loads holds 63) and measured 12 ns per position.
constexpr int kChainRing = 24;

template <int J>
__device__ __forceinline__ float lane_ahead(float v) {  // the value of the lane J places up in its row of 16
    static_assert(J >= 1 && J <= 15, "row shift");
    float r = __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(v), 0x100 + J, 0xF, 0xF, true));
    // The move stays a move (the compiler would fold it into the add as a DPP operand): an add
    // with a DPP operand has a longer latency than a plain one, and the adds are one dependent
    // chain, while the moves are independent and issue in its shadow (measured: 11 -> 8.6 cycles
    // per position).
    asm volatile("" : "+v"(r));
    return r;
}

static __global__ void __launch_bounds__(256) k_seg_chain32(const float *__restrict__ sq32,
                                                           const uint2 *__restrict__ seg_range, int dim,
                                                           float *__restrict__ var) {
    const int g = blockIdx.x;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int cb = blockIdx.y * 4 + wave;  // block of 8 columns
    if (cb * 8 >= dim) return;
    const uint2 range = seg_range[g];
    const uint32_t count = range.y - range.x;
    float acc = 0.0f;
    if (count > 0) {
        const uint32_t nP = (count + 31u) / 32u, last = nP - 1u;
        const size_t stride = (size_t)8 * dim;  // float4 per group of 32 positions
        const float4 *q = reinterpret_cast<const float4 *>(sq32 + ((size_t)range.x + 32u * (size_t)g) * dim) +
                          (size_t)cb * 64 + lane;
        // rem: positions of this group inside the segment (the same in every lane)
        auto add4 = [&](float a, float b, float c, float d, int rem, int at) {
            if (rem > at) acc = acc + a;
            if (rem > at + 1) acc = acc + b;
            if (rem > at + 2) acc = acc + c;
            if (rem > at + 3) acc = acc + d;
        };
        auto add32 = [&](const float4 &v, int rem) {
            add4(v.x, v.y, v.z, v.w, rem, 0);
            add4(lane_ahead<1>(v.x), lane_ahead<1>(v.y), lane_ahead<1>(v.z), lane_ahead<1>(v.w), rem, 4);
            add4(lane_ahead<2>(v.x), lane_ahead<2>(v.y), lane_ahead<2>(v.z), lane_ahead<2>(v.w), rem, 8);
            add4(lane_ahead<3>(v.x), lane_ahead<3>(v.y), lane_ahead<3>(v.z), lane_ahead<3>(v.w), rem, 12);
            add4(lane_ahead<4>(v.x), lane_ahead<4>(v.y), lane_ahead<4>(v.z), lane_ahead<4>(v.w), rem, 16);
            add4(lane_ahead<5>(v.x), lane_ahead<5>(v.y), lane_ahead<5>(v.z), lane_ahead<5>(v.w), rem, 20);
            add4(lane_ahead<6>(v.x), lane_ahead<6>(v.y), lane_ahead<6>(v.z), lane_ahead<6>(v.w), rem, 24);
            add4(lane_ahead<7>(v.x), lane_ahead<7>(v.y), lane_ahead<7>(v.z), lane_ahead<7>(v.w), rem, 28);
        };
        float4 buf[kChainRing];
#pragma unroll
        for (int k = 0; k < kChainRing; ++k) {
            buf[k] = q[(size_t)((uint32_t)k < last ? (uint32_t)k : last) * stride];
            // the first loads are issued in slot order, as the loop issues them: the loop's waits count
            // the loads issued after a slot's, and one order on both ways into the loop keeps them exact
            asm volatile("" ::: "memory");
        }
        const uint32_t full = count / 32u;  // groups with all their positions
        uint32_t P = 0;
        for (; P + kChainRing <= full; P += kChainRing) {
#pragma unroll
            for (int k = 0; k < kChainRing; ++k) {
                // (added first, refilled after: the slot's register is free when its load is issued,
                // so no copy of the ring is carried around the loop)
                add32(buf[k], 32);
                const uint32_t nx = P + kChainRing + k;
                buf[k] = q[(size_t)(nx < last ? nx : last) * stride];
            }
        }
#pragma unroll
        for (int k = 0; k < kChainRing; ++k) {
            const int rem = (int)count - 32 * (int)(P + k);
            if (rem > 0) add32(buf[k], rem);
        }
    }
    if ((lane & 7) == 0) var[(size_t)g * dim + cb * 8 + (lane >> 3)] = acc;
}

// ---- the same sequential sums without the long chain -------------------------------------------
// A sequential f32 sum of non-negative terms is, while the running sum S stays inside one binade
// [2^e, 2^(e+1)], an integer accumulation: with u = 2^(e-23) and S = s u, fl(S + t) = (s + r) u where
// r is t / u rounded to an integer, to nearest, a tie to the value that makes s + r even.  So a
// group of 32 terms acts on s as s -> s + inc[parity of s], two integers per group that depend on e
// only, and the maps of consecutive groups compose.  Three steps on top of k_seg_sqdev32 (which
// also emits every group's approximate sum):
//   k_seg_chain_guess    per column, a prefix over the group sums in f64 gives the binade the running
//                        sum will be in at each group (two candidates near a boundary)
//   k_seg_chain_maps     per (group, column), on the whole GPU: inc[0], inc[1] for the guessed binade(s)
//   k_seg_chain_compose  per column, one wave: 64 groups at a time, the maps composed by a scan over
//                        the lanes; it checks every assumption (S is in the guessed binade at the
//                        group's start and does not leave it) and adds a group's 32 terms one by one
//                        where one fails — the groups in which S crosses a binade, the first groups,
//                        non-finite values.  The result is the sequential sum, bit for bit.
// The value of the lane K places down in its row of 16 lanes (DPP row shift), `fill` where that lane
// is outside the row: scans over the wave take four of these steps and three broadcasts of a row's
// last lane instead of six permutes through LDS.
template <int K>
__device__ __forceinline__ uint32_t row_shr(uint32_t v, uint32_t fill) {
    return (uint32_t)__builtin_amdgcn_update_dpp((int)fill, (int)v, 0x110 + K, 0xF, 0xF, false);
}
template <int K>
__device__ __forceinline__ double row_shr_f64(double v) {  // 0.0 where the lane is outside the row
    const unsigned long long b = (unsigned long long)__double_as_longlong(v);
    const uint32_t lo = row_shr<K>((uint32_t)b, 0u), hi = row_shr<K>((uint32_t)(b >> 32), 0u);
    return __longlong_as_double((long long)(((unsigned long long)hi << 32) | lo));
}
__device__ __forceinline__ double lane_f64(double v, int src) {  // src: a constant lane
    const unsigned long long b = (unsigned long long)__double_as_longlong(v);
    const uint32_t lo = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)b, src);
    const uint32_t hi = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)(b >> 32), src);
    return __longlong_as_double((long long)(((unsigned long long)hi << 32) | lo));
}

constexpr uint32_t kMapInvalid = 0xFFFFFFFFu;
// guess code: exponent field of the lower candidate | two candidates | all terms zero | usable
constexpr uint16_t kGuessOk = 0x8000u, kGuessTwo = 0x0100u, kGuessZero = 0x0200u;

// Long columns are cut into blocks of kGuessBlock groups that are guessed side by side: the f64 sum
// of every block first (grid (segments, dim / 4, blocks); 4 waves, one column each), then a block's
// prefix starts from the sum of the blocks before it.
constexpr uint32_t kGuessBlock = 1024;
static __global__ void __launch_bounds__(256) k_seg_chain_bsum(const float *__restrict__ gsum,
                                                              const uint2 *__restrict__ seg_range, int dim,
                                                              double *__restrict__ bsum) {
    const int g = blockIdx.x, lane = threadIdx.x & 63, c = blockIdx.y * 4 + (threadIdx.x >> 6);
    if (c >= dim) return;
    const uint2 range = seg_range[g];
    const uint32_t count = range.y - range.x, nP = (count + 31u) / 32u;
    const uint32_t P0 = blockIdx.z * kGuessBlock;
    if (P0 >= nP) return;
    const size_t g0 = seg_group0(range, g);
    float vin[16];
#pragma unroll
    for (int k = 0; k < 16; ++k) {
        const uint32_t P = P0 + 64 * k + lane;
        vin[k] = gsum[(g0 + (P < nP ? P : nP - 1)) * dim + c];
    }
    double acc = 0.0;
#pragma unroll
    for (int k = 0; k < 16; ++k) acc += (P0 + 64 * k + lane < nP) ? (double)vin[k] : 0.0;
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) acc += __shfl_xor(acc, off);
    if (lane == 0) bsum[((size_t)g * gridDim.z + blockIdx.z) * dim + c] = acc;
}

// grid (segments, dim / 4, blocks); 256 threads = 4 waves, one column each.  bsum == nullptr: one
// block per column, whatever its length.
static __global__ void __launch_bounds__(256) k_seg_chain_guess(const float *__restrict__ gsum,
                                                               const uint2 *__restrict__ seg_range, int dim,
                                                               const double *__restrict__ bsum,
                                                               uint16_t *__restrict__ guess) {
    const int g = blockIdx.x, lane = threadIdx.x & 63, c = blockIdx.y * 4 + (threadIdx.x >> 6);
    if (c >= dim) return;
    const uint2 range = seg_range[g];
    const uint32_t count = range.y - range.x, nP_all = (count + 31u) / 32u;
    const size_t g0 = seg_group0(range, g);
    double carry = 0.0;
    uint32_t P_first = 0, nP = nP_all;
    if (bsum) {
        P_first = blockIdx.z * kGuessBlock;
        if (P_first >= nP_all) return;
        nP = nP_all - P_first < kGuessBlock ? nP_all : P_first + kGuessBlock;
        for (uint32_t b = lane; b < blockIdx.z; b += 64) carry += bsum[((size_t)g * gridDim.z + b) * dim + c];
#pragma unroll
        for (int off = 32; off > 0; off >>= 1) carry += __shfl_xor(carry, off);
    }
    constexpr int R = 16;  // batches of 64 groups per round of loads (one memory round trip per round)
    for (uint32_t P0 = P_first; P0 < nP; P0 += 64 * R) {
        float vin[R];
#pragma unroll
        for (int k = 0; k < R; ++k) {
            const uint32_t P = P0 + 64 * k + lane;
            vin[k] = gsum[(g0 + (P < nP ? P : nP - 1)) * dim + c];
        }
#pragma unroll
        for (int k = 0; k < R; ++k) {
            const uint32_t P = P0 + 64 * k + lane;
            const double v = P < nP ? (double)vin[k] : 0.0;
            // inclusive prefix over the lanes: inside the rows of 16, then row by row
            double inc = v;
            inc += row_shr_f64<1>(inc);
            inc += row_shr_f64<2>(inc);
            inc += row_shr_f64<4>(inc);
            inc += row_shr_f64<8>(inc);
            {
                const double r0 = lane_f64(inc, 15);
                if ((lane >> 4) == 1) inc += r0;
                const double r1 = lane_f64(inc, 31);
                if ((lane >> 4) == 2) inc += r1;
                const double r2 = lane_f64(inc, 47);
                if ((lane >> 4) == 3) inc += r2;
            }
            const double before = carry + (inc - v), after = carry + inc;
            carry = lane_f64(after, 63);
            if (P < nP) {
                // the sequential f32 sum is within 2^-9 of the f64 one by a wide margin
                const float lo = (float)(before * (1.0 - 0.001953125)), hi = (float)(after * (1.0 + 0.001953125));
                const uint32_t elo = __float_as_uint(lo) >> 23, ehi = __float_as_uint(hi) >> 23;  // both >= +0
                uint16_t code = 0;
                if (v == 0.0)  // non-negative terms with a zero sum: every one is +0 and leaves any S as it is
                    code = (uint16_t)(kGuessOk | kGuessZero);
                else if (before > 0.0 && elo >= 30u && ehi <= 250u && ehi - elo <= 1u)
                    code = (uint16_t)(kGuessOk | (ehi != elo ? kGuessTwo : 0u) | elo);
                guess[(g0 + P) * dim + c] = code;
            }
        }
    }
}

// inc[0], inc[1] of one group for a running sum in the binade of exponent field e (30 <= e <= 250).
// A term over the unit, y = t / u = t * 2^(150 - e), is exact (a scaling by a power of two; a product
// that underflows stays below 1/2 and counts as zero either way), so its integer part, and whether
// the rest is above or exactly one half, come from a floor and a subtraction, both exact below 2^24.
__device__ __forceinline__ void chain_group_map(const float (&t)[32], int valid, uint32_t e, uint32_t &inc0,
                                                uint32_t &inc1) {
    const float inv_u = __uint_as_float((277u - e) << 23);  // 2^(150 - e)
    // s0, s1: the running sum's integer for an even and for an odd start, less the (even) start
    // itself: their lowest bits are the parities the tie rule asks for
    uint32_t s0 = 0, s1 = 1;
    bool bad = false;
#pragma unroll
    for (int i = 0; i < 32; ++i) {
        if (i < valid) {
            const float y = t[i] * inv_u;
            // a negative term, a NaN, an infinity, or a term of a higher binade than the sum's
            bad = bad || !(y >= 0.0f) || !(y < 16777216.0f);
            const float f = floorf(y);
            const float rest = y - f;
            const uint32_t q = (uint32_t)f;
            const uint32_t tie = rest == 0.5f ? 1u : 0u;
            const uint32_t step = q + (rest > 0.5f ? 1u : 0u);
            // a tie goes up when that makes the sum even: when sum + q is odd
            s0 += step + (tie & (s0 + q));
            s1 += step + (tie & (s1 + q));
        }
    }
    inc0 = bad ? kMapInvalid : s0;
    inc1 = bad ? kMapInvalid : s1 - 1u;
}

// Grid (blocks of 64 positions, segments), as k_seg_sqdev32: one thread per (group, column).
static __global__ void __launch_bounds__(256) k_seg_chain_maps(const uint32_t *__restrict__ perm,
                                                              const uint2 *__restrict__ seg_range,
                                                              const float *__restrict__ means, int64_t first,
                                                              const float *__restrict__ x, int64_t ld, int dim,
                                                              const uint16_t *__restrict__ guess,
                                                              uint4 *__restrict__ maps) {
    const int g = blockIdx.y;
    const uint2 range = seg_range[g];
    const uint32_t count = range.y - range.x;
    const uint32_t P0 = blockIdx.x * 2u;
    if (P0 * 32u >= count) return;
    const uint32_t nP = (count + 31u) / 32u;
    const uint32_t groups = nP - P0 < 2u ? nP - P0 : 2u;
    const float *mrow = means + (first + g) * dim;
    const uint32_t *pm = perm + range.x;
    const size_t g0 = seg_group0(range, g);
    for (uint32_t e = threadIdx.x; e < groups * (uint32_t)dim; e += 256) {
        const uint32_t P = P0 + e / (uint32_t)dim, c = e % (uint32_t)dim;
        const uint16_t code = guess[(g0 + P) * dim + c];
        uint4 out = make_uint4(kMapInvalid, kMapInvalid, kMapInvalid, kMapInvalid);
        if (code & kGuessZero) {
            out = make_uint4(0u, 0u, 0u, 0u);
        } else if (code & kGuessOk) {
            // the squares again, with the same two roundings (past the end: the last row, not counted)
            const float m = mrow[c];
            float t[32];
#pragma unroll
            for (int r = 0; r < 32; ++r) {
                const uint32_t p = 32u * P + r;
                const float d = x[(int64_t)pm[p < count ? p : count - 1] * ld + c] - m;
                t[r] = d * d;
            }
            const int valid = (int)(count - 32u * P < 32u ? count - 32u * P : 32u);
            const uint32_t elo = code & 255u;
            chain_group_map(t, valid, elo, out.x, out.y);
            if (code & kGuessTwo) chain_group_map(t, valid, elo + 1u, out.z, out.w);
        }
        maps[(g0 + P) * dim + c] = out;
    }
}

// The map of the lanes' groups composed over the wave: on return lane p holds the map of the groups
// of lanes first .. p (lanes outside [first, last) supply the identity), as increments for an even
// and for an odd start, saturated at 2^25.
__device__ __forceinline__ void chain_scan_maps(uint32_t &a0, uint32_t &a1, int lane) {
    const uint32_t cap = 1u << 25;
    // left, then this lane's map: c_p = l_p + a_[(p + l_p) mod 2]; (0, 0) is the identity, which is what a
    // lane outside the row supplies
    auto after_left = [&](uint32_t l0, uint32_t l1) {
        const uint32_t n0 = l0 + ((l0 & 1u) ? a1 : a0);        // start even: after l0 the parity is l0 & 1
        const uint32_t n1 = l1 + (((l1 + 1u) & 1u) ? a1 : a0);  // start odd
        a0 = n0 < cap ? n0 : cap;
        a1 = n1 < cap ? n1 : cap;
    };
    after_left(row_shr<1>(a0, 0u), row_shr<1>(a1, 0u));
    after_left(row_shr<2>(a0, 0u), row_shr<2>(a1, 0u));
    after_left(row_shr<4>(a0, 0u), row_shr<4>(a1, 0u));
    after_left(row_shr<8>(a0, 0u), row_shr<8>(a1, 0u));
    uint32_t t0 = (uint32_t)__builtin_amdgcn_readlane((int)a0, 15), t1 = (uint32_t)__builtin_amdgcn_readlane((int)a1, 15);
    if ((lane >> 4) == 1) after_left(t0, t1);
    t0 = (uint32_t)__builtin_amdgcn_readlane((int)a0, 31), t1 = (uint32_t)__builtin_amdgcn_readlane((int)a1, 31);
    if ((lane >> 4) == 2) after_left(t0, t1);
    t0 = (uint32_t)__builtin_amdgcn_readlane((int)a0, 47), t1 = (uint32_t)__builtin_amdgcn_readlane((int)a1, 47);
    if ((lane >> 4) == 3) after_left(t0, t1);
}

// Runs of kRunGroups consecutive groups of a long column get their maps composed ahead of the walk
// (k_seg_chain_runs): a run is "clean" when every group has one guessed binade, the same in all of
// them (groups of zeros fit any), and a usable map.  The walk then passes a clean run in one step
// when S is in that binade at the run's start and does not leave it by the run's end — S never
// decreases, so it is in the binade at every group in between and each group's map applies, which is
// all the group-by-group walk checks.  Any other run is walked group by group as before.
constexpr uint32_t kRunGroups = 256;
constexpr uint32_t kRunClean = 0x80000000u, kRunAnyBinade = 0x40000000u;

// Index of a segment's first run in the per-run table (runs of different segments never share one).
__device__ __forceinline__ size_t seg_run0(const uint2 range, int g) {
    return seg_group0(range, g) / kRunGroups + (size_t)g;
}

// grid (segments, dim / 4, ceil(groups / 1024)); 256 threads = 4 waves, one column each; a wave
// composes four runs (16 batches of 64 groups, one round of loads).
static __global__ void __launch_bounds__(256) k_seg_chain_runs(const uint2 *__restrict__ seg_range, int dim,
                                                              const uint16_t *__restrict__ guess,
                                                              const uint4 *__restrict__ maps,
                                                              uint4 *__restrict__ runs) {
    const int g = blockIdx.x, lane = threadIdx.x & 63, c = blockIdx.y * 4 + (threadIdx.x >> 6);
    if (c >= dim) return;
    const uint2 range = seg_range[g];
    const uint32_t count = range.y - range.x, nP = (count + 31u) / 32u;
    const uint32_t P0 = blockIdx.z * (4u * kRunGroups);
    if (P0 >= nP) return;
    const size_t g0 = seg_group0(range, g), r0 = seg_run0(range, g);
    constexpr int R = 16;
    uint16_t codeR[R];
    uint4 mpR[R];
#pragma unroll
    for (int k = 0; k < R; ++k) {
        const uint32_t idx = P0 + 64u * k + lane;
        const size_t at = (g0 + (idx < nP ? idx : nP - 1u)) * dim + c;
        codeR[k] = guess[at];
        mpR[k] = maps[at];
    }
    const uint32_t cap = 1u << 25;
#pragma unroll
    for (int run = 0; run < 4; ++run) {
        const uint32_t Pr = P0 + run * kRunGroups;
        if (Pr >= nP) break;  // uniform
        uint32_t c0 = 0, c1 = 0, e = 0;
        bool clean = true, any_binade = true;
#pragma unroll
        for (int k4 = 0; k4 < 4; ++k4) {
            const int k = 4 * run + k4;
            const uint32_t base = Pr + 64u * k4;
            const uint32_t left = base >= nP ? 0u : (nP - base < 64u ? nP - base : 64u);
            if (left == 0u) break;  // uniform
            const uint16_t code = codeR[k];
            const uint4 mp = mpR[k];
            const bool mine = (uint32_t)lane < left;
            const bool zero = (code & kGuessZero) != 0;
            const uint32_t elo = code & 255u;
            const bool usable = (code & kGuessOk) &&
                                (zero || (!(code & kGuessTwo) && mp.x != kMapInvalid && elo >= 30u && elo <= 250u));
            if (__ballot(mine && !usable)) clean = false;
            const unsigned long long binade = __ballot(mine && !zero);
            if (binade) {
                const uint32_t ef = (uint32_t)__builtin_amdgcn_readlane((int)elo, __ffsll((long long)binade) - 1);
                if (any_binade) e = ef;
                any_binade = false;
                if (__ballot(mine && !zero && elo != e)) clean = false;
            }
            uint32_t a0 = (mine && !zero) ? (mp.x < cap ? mp.x : cap) : 0u;
            uint32_t a1 = (mine && !zero) ? (mp.y < cap ? mp.y : cap) : 0u;
            chain_scan_maps(a0, a1, lane);
            const uint32_t b0 = (uint32_t)__builtin_amdgcn_readlane((int)a0, 63), b1 = (uint32_t)__builtin_amdgcn_readlane((int)a1, 63);
            // the run so far, then this batch
            const uint32_t n0 = c0 + ((c0 & 1u) ? b1 : b0), n1 = c1 + (((c1 + 1u) & 1u) ? b1 : b0);
            c0 = n0 < cap ? n0 : cap;
            c1 = n1 < cap ? n1 : cap;
        }
        if (lane == 0)
            runs[(r0 + Pr / kRunGroups) * dim + c] =
                make_uint4(c0, c1, (clean ? kRunClean : 0u) | (any_binade ? kRunAnyBinade : 0u) | e, 0u);
    }
}

// One batch of up to 64 groups (lane = group base + lane) added to S, which is the same value in every
// lane: runs of usable groups through their composed maps, any other group term by term.
__device__ __forceinline__ void chain_batch(float &S, uint32_t base, uint32_t left, uint16_t code, uint4 mp,
                                            const uint32_t *__restrict__ pm, uint32_t count,
                                            const float *__restrict__ x, int64_t ld, int c, float mean_c, int lane) {
    const uint32_t elo = code & 255u;
    const bool zero = (code & kGuessZero) != 0;
    uint32_t start = 0;  // groups of the batch already added
    while (start < left) {
        // S is +0, positive, +inf or a NaN; with the sign bit of a NaN eS is above every guess
        const uint32_t Sb = __float_as_uint(S), eS = Sb >> 23;
        const uint32_t s = (Sb & 0x7fffffu) | 0x800000u;  // S / u for a normal S
        const bool is_lo = elo == eS, is_hi = (code & kGuessTwo) && elo + 1u == eS;
        uint32_t a0 = is_lo ? mp.x : mp.z, a1 = is_lo ? mp.y : mp.w;
        // a group of zeros keeps any finite S; another group needs S in the binade of its map
        const bool mine = (uint32_t)lane >= start && (uint32_t)lane < left;
        const bool ok = (code & kGuessOk) &&
                        (zero ? eS < 255u : (eS >= 30u && eS <= 250u && (is_lo || is_hi) && a0 != kMapInvalid));
        if (zero) a0 = a1 = 0u;
        // the run of usable groups that starts at `start`
        const unsigned long long stop = __ballot(mine && !ok) | (left < 64u ? ~0ull << left : 0ull);
        const uint32_t end = stop ? (uint32_t)__ffsll((long long)stop) - 1u : 64u;
        bool advanced = false;
        if (end > start) {
            const uint32_t cap = 1u << 25;
            const bool part = (uint32_t)lane >= start && (uint32_t)lane < end;
            a0 = part ? (a0 < cap ? a0 : cap) : 0u;
            a1 = part ? (a1 < cap ? a1 : cap) : 0u;
            // inclusive scan: the map of groups start .. lane, as increments for a start parity
            chain_scan_maps(a0, a1, lane);
            const uint32_t send = s + ((s & 1u) ? a1 : a0);
            const bool fits = part && send <= (1u << 24);
            const int nv = __popcll(__ballot(fits));  // fits is monotone: the sums never decrease
            if (nv > 0) {
                const uint32_t take = (uint32_t)__builtin_amdgcn_readlane((int)send, __builtin_amdgcn_readfirstlane((int)start + nv - 1));
                // (a subnormal or zero S only passes groups of zeros: take == s and S stays)
                S = __uint_as_float(take == (1u << 24) ? (eS + 1u) << 23 : (eS << 23) | (take - (1u << 23)));
                start += (uint32_t)nv;
                advanced = true;
            }
        }
        if (!advanced) {
            // the group's terms one by one (positions past the end add +0.0, which changes nothing)
            const uint32_t P = base + start;
            float t = 0.0f;
            if (lane < 32 && P * 32u + (uint32_t)lane < count) {
                const float d = x[(int64_t)pm[P * 32u + lane] * ld + c] - mean_c;
                t = d * d;
            }
#pragma unroll
            for (int i = 0; i < 32; ++i) S = S + __shfl(t, i);
            start += 1u;
        }
    }
}

// grid (segments, dim / 4); 256 threads = 4 waves, one column each.  runs == nullptr: every group is
// walked (short columns); else the table of k_seg_chain_runs.
static __global__ void __launch_bounds__(256) k_seg_chain_compose(const uint32_t *__restrict__ perm,
                                                                 const uint2 *__restrict__ seg_range,
                                                                 const float *__restrict__ means, int64_t first,
                                                                 const float *__restrict__ x, int64_t ld, int dim,
                                                                 const uint16_t *__restrict__ guess,
                                                                 const uint4 *__restrict__ maps,
                                                                 const uint4 *__restrict__ runs,
                                                                 float *__restrict__ var) {
    const int g = blockIdx.x, lane = threadIdx.x & 63, c = blockIdx.y * 4 + (threadIdx.x >> 6);
    if (c >= dim) return;
    const uint2 range = seg_range[g];
    const uint32_t count = range.y - range.x, nP = (count + 31u) / 32u;
    const size_t g0 = seg_group0(range, g);
    const float mean_c = means[(first + g) * dim + c];
    const uint32_t *pm = perm + range.x;
    float S = 0.0f;  // the same value in every lane
    if (runs) {
        const size_t r0 = seg_run0(range, g);
        const uint32_t nR = (nP + kRunGroups - 1u) / kRunGroups;
        for (uint32_t rb = 0; rb < nR; rb += 64) {
            const uint32_t ri = rb + lane;
            const uint4 rm = runs[(r0 + (ri < nR ? ri : nR - 1u)) * dim + c];  // lane = run rb + lane
            const uint32_t here = nR - rb < 64u ? nR - rb : 64u;
            for (uint32_t j = 0; j < here; ++j) {
                const uint32_t c0 = (uint32_t)__builtin_amdgcn_readlane((int)rm.x, (int)j);
                const uint32_t c1 = (uint32_t)__builtin_amdgcn_readlane((int)rm.y, (int)j);
                const uint32_t meta = (uint32_t)__builtin_amdgcn_readlane((int)rm.z, (int)j);
                const uint32_t Sb = __float_as_uint(S), eS = Sb >> 23;
                const uint32_t s = (Sb & 0x7fffffu) | 0x800000u;
                const uint32_t send = s + ((s & 1u) ? c1 : c0);
                const bool binade_ok = (meta & kRunAnyBinade) ? eS < 255u : (eS == (meta & 255u) && eS >= 30u && eS <= 250u);
                if ((meta & kRunClean) && binade_ok && send <= (1u << 24)) {
                    // (a run of zeros: send == s and S stays, whatever finite value it has)
                    if (!(meta & kRunAnyBinade))
                        S = __uint_as_float(send == (1u << 24) ? (eS + 1u) << 23 : (eS << 23) | (send - (1u << 23)));
                    continue;
                }
                // group by group: the run's four batches
                const uint32_t Pr = (rb + j) * kRunGroups;
                uint16_t codeR[4];
                uint4 mpR[4];
#pragma unroll
                for (int k = 0; k < 4; ++k) {
                    const uint32_t idx = Pr + 64u * k + lane;
                    const size_t at = (g0 + (idx < nP ? idx : nP - 1u)) * dim + c;
                    codeR[k] = guess[at];
                    mpR[k] = maps[at];
                }
#pragma unroll
                for (int k = 0; k < 4; ++k) {
                    const uint32_t base = Pr + 64u * k;
                    const uint32_t left = base >= nP ? 0u : (nP - base < 64u ? nP - base : 64u);
                    chain_batch(S, base, left, codeR[k], mpR[k], pm, count, x, ld, c, mean_c, lane);
                }
            }
        }
        if (lane == 0) var[(size_t)g * dim + c] = S;
        return;
    }
    // Batches of 64 groups at fixed positions (lane = group 64 b + lane), R batches per round of
    // loads: one memory round trip per round instead of one per batch.
    constexpr int R = 16;
    const uint32_t nB = (nP + 63u) / 64u;
    for (uint32_t b0 = 0; b0 < nB; b0 += R) {
        uint16_t codeR[R];
        uint4 mpR[R];
#pragma unroll
        for (int k = 0; k < R; ++k) {
            const uint32_t idx = (b0 + k) * 64u + lane;
            const size_t at = (g0 + (idx < nP ? idx : nP - 1u)) * dim + c;
            codeR[k] = guess[at];
            mpR[k] = maps[at];
        }
#pragma unroll
        for (int k = 0; k < R; ++k) {
            const uint32_t base = (b0 + k) * 64u;  // first group of the batch
            // groups in the batch (none past the end: the loop inside does not run; uniform)
            const uint32_t left = base >= nP ? 0u : (nP - base < 64u ? nP - base : 64u);
            chain_batch(S, base, left, codeR[k], mpR[k], pm, count, x, ld, c, mean_c, lane);
        }
    }
    if (lane == 0) var[(size_t)g * dim + c] = S;
}

__device__ __forceinline__ void lds_only_barrier() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

__device__ __forceinline__ int find_segment(const uint2 *__restrict__ seg_range, int nseg, uint32_t p) {
    // segments are sorted by position and disjoint; returns -1 when p lies in none
    int lo = 0, hi = nseg - 1;
    while (lo <= hi) {
        int mid = (lo + hi) >> 1;
        uint2 r = seg_range[mid];
        if (p < r.x)
            hi = mid - 1;
        else if (p >= r.y)
            lo = mid + 1;
        else
            return mid;
    }
    return -1;
}

// vals[p] = x[perm[p]][split_dim[segment of p]]; positions outside every segment get +inf
static __global__ void __launch_bounds__(256) k_seg_gather_col(const uint32_t *__restrict__ perm, int64_t n,
                                                        const uint2 *__restrict__ seg_range, int nseg,
                                                        const int *__restrict__ split_dim,
                                                        const float *__restrict__ x, int64_t ld,
                                                        float *__restrict__ vals) {
    int64_t p = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (p >= n) return;
    int g = find_segment(seg_range, nseg, (uint32_t)p);
    vals[p] = g < 0 ? __builtin_inff() : x[(int64_t)perm[p] * ld + split_dim[g]];
}

// flags[p] = 1 when the row at position p goes left (value <= median of its segment)
static __global__ void __launch_bounds__(256) k_seg_flags(const float *__restrict__ vals, int64_t n,
                                                   const uint2 *__restrict__ seg_range, int nseg,
                                                   const float *__restrict__ median,
                                                   uint32_t *__restrict__ flags) {
    int64_t p = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (p >= n) return;
    int g = find_segment(seg_range, nseg, (uint32_t)p);
    flags[p] = (g >= 0 && vals[p] <= median[g]) ? 1u : 0u;
}

// Stable partition inside every segment using the exclusive scan of flags.
// nleft[g] = number of rows going left.
static __global__ void __launch_bounds__(256) k_seg_partition(const uint32_t *__restrict__ perm_in, int64_t n,
                                                       const uint2 *__restrict__ seg_range, int nseg,
                                                       const uint32_t *__restrict__ flags,
                                                       const uint32_t *__restrict__ scan,
                                                       uint32_t *__restrict__ perm_out,
                                                       uint32_t *__restrict__ nleft) {
    int64_t p = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (p >= n) return;
    int g = find_segment(seg_range, nseg, (uint32_t)p);
    if (g < 0) {
        perm_out[p] = perm_in[p];
        return;
    }
    uint2 r = seg_range[g];
    uint32_t before = scan[p] - scan[r.x];                       // left rows before p in the segment
    uint32_t total_left = scan[r.y - 1] + flags[r.y - 1] - scan[r.x];
    uint32_t dst = flags[p] ? r.x + before : r.x + total_left + ((uint32_t)p - r.x - before);
    perm_out[dst] = perm_in[p];
    if ((uint32_t)p == r.x) nleft[g] = total_left;
}

static __global__ void __launch_bounds__(256) k_iota_u32(uint32_t *__restrict__ p, int64_t n) {
    int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (i < n) p[i] = (uint32_t)i;
}

// ---- middle values by radix select ---------------------------------------------------------
// The reference sorts the split column and takes values[c/2] (and values[c/2 - 1] for an even
// count, src/tsvq.rs:108-117); only those two order statistics are needed.  Floats are mapped to
// unsigned keys of the same order; four passes of 8 bits narrow each target down: a pass counts,
// per segment and target, the keys that share the target's known high bits by their next byte
// (LDS histograms per workgroup, flushed with integer atomics), then one thread per (segment,
// target) picks the byte whose bin holds the target's rank.
struct SegSelect {
    uint32_t prefix;  // known high bits of the key (low bits zero)
    uint32_t rank;    // rank of the target among the keys that share the prefix
};

__device__ __forceinline__ uint32_t float_order_key(float f) {
    const uint32_t u = __float_as_uint(f);
    return (u & 0x80000000u) ? ~u : (u | 0x80000000u);
}
__device__ __forceinline__ float float_from_order_key(uint32_t k) {
    return __uint_as_float((k & 0x80000000u) ? (k & 0x7fffffffu) : ~k);
}

// One workgroup per 4096 positions; pass = 0..3 looks at key bits [31 - 8 pass, 24 - 8 pass].
static __global__ void __launch_bounds__(256) k_seg_select_hist(const float *__restrict__ vals, int64_t n,
                                                                const uint2 *__restrict__ seg_range, int nseg,
                                                                const SegSelect *__restrict__ sel, int pass,
                                                                uint32_t *__restrict__ hist) {
    __shared__ uint32_t lh[512];
    const int64_t lo = (int64_t)blockIdx.x * 4096;
    const int64_t hi = lo + 4096 < n ? lo + 4096 : n;
    const int shift = 24 - 8 * pass;
    const uint32_t high_mask = pass == 0 ? 0u : (0xFFFFFFFFu << (shift + 8));
    // segments are sorted by position and disjoint: walk the ones that overlap this chunk
    int g = 0;
    {
        int a = 0, b = nseg;  // first segment whose end is beyond lo
        while (a < b) {
            const int mid = (a + b) >> 1;
            if (seg_range[mid].y <= (uint32_t)lo) a = mid + 1; else b = mid;
        }
        g = a;
    }
    for (; g < nseg; ++g) {
        const uint2 r = seg_range[g];
        if ((int64_t)r.x >= hi) break;
        const int64_t from = (int64_t)r.x > lo ? (int64_t)r.x : lo, to = (int64_t)r.y < hi ? (int64_t)r.y : hi;
        const uint32_t p0 = sel[2 * g].prefix, p1 = sel[2 * g + 1].prefix;
        __syncthreads();
        lh[threadIdx.x] = 0u;
        lh[256 + threadIdx.x] = 0u;
        __syncthreads();
        for (int64_t p = from + threadIdx.x; p < to; p += 256) {
            const uint32_t key = float_order_key(vals[p]);
            const uint32_t byte = (key >> shift) & 255u;
            if ((key & high_mask) == p0) atomicAdd(&lh[byte], 1u);
            if ((key & high_mask) == p1) atomicAdd(&lh[256 + byte], 1u);
        }
        __syncthreads();
        uint32_t *gh = hist + (size_t)g * 512;
        if (lh[threadIdx.x]) atomicAdd(&gh[threadIdx.x], lh[threadIdx.x]);
        if (lh[256 + threadIdx.x]) atomicAdd(&gh[256 + threadIdx.x], lh[256 + threadIdx.x]);
    }
}

// One wave per (segment, target): the byte whose bin holds the rank; clears the bins.  A lane
// takes four bins, a scan over the lanes finds the one whose bins hold the rank.
static __global__ void __launch_bounds__(64) k_seg_select_pick(uint32_t *__restrict__ hist,
                                                               SegSelect *__restrict__ sel, int nseg, int pass) {
    const int i = blockIdx.x, lane = threadIdx.x;
    if (i >= 2 * nseg) return;
    uint4 *h = reinterpret_cast<uint4 *>(hist + (size_t)i * 256);
    const uint4 c = h[lane];
    h[lane] = make_uint4(0u, 0u, 0u, 0u);
    const SegSelect s = sel[i];
    const uint32_t tot = c.x + c.y + c.z + c.w;
    uint32_t inc = tot;
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
        const uint32_t v = __shfl_up(inc, off);
        if (lane >= off) inc += v;
    }
    const uint32_t exc = inc - tot;
    const bool mine = s.rank >= exc && s.rank < inc;
    const int shift = 24 - 8 * pass;
    if (mine) {
        uint32_t r = s.rank - exc, byte = 4u * (uint32_t)lane;
        if (r >= c.x) {
            r -= c.x;
            ++byte;
            if (r >= c.y) {
                r -= c.y;
                ++byte;
                if (r >= c.z) {
                    r -= c.z;
                    ++byte;
                }
            }
        }
        sel[i] = SegSelect{s.prefix | (byte << shift), r};
    }
    // a rank beyond the counted keys (never for a rank inside its segment): the last byte
    const uint32_t all = __shfl(inc, 63);
    if (lane == 0 && s.rank >= all) sel[i] = SegSelect{s.prefix | (255u << shift), s.rank - all};
}

// The split dimension of every segment: argmax of its per-dimension sums with the LAST maximal
// element winning (Iterator::max_by, src/tsvq.rs:102-106); one thread per segment.
// The same launch starts the radix select of the middle values: bins cleared, ranks of the two
// targets of every segment (the lower and the upper middle).  Grid over nseg * 512 bins.
// var: rows of `stride` values, the first dim of them the row's components (padded rows: zeros behind them).
static __global__ void k_seg_argmax_last(const float *__restrict__ var, int nseg, int dim, int stride, int *__restrict__ sdim,
                                         const uint2 *__restrict__ seg_range, SegSelect *__restrict__ sel,
                                         uint32_t *__restrict__ hist) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < nseg * 512) hist[i] = 0u;
    if (i >= nseg) return;
    {
        const uint2 r = seg_range[i];
        const uint32_t c = r.y - r.x;
        sel[2 * i] = SegSelect{0u, (c % 2 == 0) ? c / 2 - 1 : c / 2};
        sel[2 * i + 1] = SegSelect{0u, c / 2};
    }
    const float *v = var + (size_t)i * stride;
    int best = 0;
    float vb = v[0];
    for (int t0 = 1; t0 < dim; t0 += 16) {
        float w[16];  // sixteen loads in flight
#pragma unroll
        for (int u = 0; u < 16; ++u) w[u] = v[t0 + u < dim ? t0 + u : dim - 1];
#pragma unroll
        for (int u = 0; u < 16; ++u) {
            if (t0 + u < dim && !(w[u] < vb)) {
                best = t0 + u;
                vb = w[u];
            }
        }
    }
    sdim[i] = best;
}

// The median of every segment from its two middle values (src/tsvq.rs:112-117): their f32 sum
// divided by two for an even count, the middle value otherwise.
static __global__ void k_seg_median(const SegSelect *__restrict__ sel, const uint2 *__restrict__ seg_range, int nseg,
                                    float *__restrict__ median) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= nseg) return;
    const uint32_t cnt = seg_range[i].y - seg_range[i].x;
    // the selected keys back as floats
    const float a = float_from_order_key(sel[2 * i].prefix), b = float_from_order_key(sel[2 * i + 1].prefix);
    const float sum = a + b;
    median[i] = (cnt % 2u == 0u) ? sum / 2.0f : a;
}

// Split dimension, median and stable partition of one node by one workgroup, for levels whose nodes all fit
// LDS: k_seg_argmax_last ... k_seg_partition are fourteen launches with the host's launch times between
// them (100-150 us per level of 100,000 rows), whatever the nodes' sizes; this is one of 45 us (8 nodes of 12,500
// rows) to 9 us (512 nodes).
// lds: the keys of the node's rows, 2 x 256 counters, the waves' partial sums.  Any number of whole waves.
constexpr uint32_t kSplitWgMax = 16384;  // rows: 64 KB of keys
inline size_t split_wg_lds(uint32_t longest) { return sizeof(uint32_t) * ((size_t)longest + 512 + 64); }

// One node of a workgroup: v its per-dimension sums, r its positions in perm, key room for its rows' keys (LDS or
// memory).  Split dimension, median and left count through the pointers (thread 0).  Returns the left count.
__device__ __forceinline__ uint32_t split_node(uint32_t *hist, uint32_t *part, uint32_t *key, const uint32_t *__restrict__ perm, const uint2 r,
                                               const float *__restrict__ v, int dim, const float *__restrict__ x, int64_t ld,
                                               int *split_dim, float *median, uint32_t *nleft, uint32_t *__restrict__ perm_out) {
    const int tid = threadIdx.x, nt = blockDim.x, lane = tid & 63, wave = tid >> 6, nw = nt >> 6;
    const uint32_t cnt = r.y - r.x;
    // The reference's scan keeps an index for which !(v[t] < best so far): the last of the largest values, and a
    // NaN or what follows one is always taken.  A run of values acts on what came before as its own result
    // does, unless it holds a NaN: then it decides alone; so runs compose in order, one per lane.
    if (wave == 0) {
        const int per = (dim + 63) / 64, t0 = lane * per, t1 = t0 + per < dim ? t0 + per : dim;
        int best = t0;
        float vb = t0 < dim ? v[t0] : 0.0f;
        bool any = t0 < dim, alone = any && !(vb == vb);
        for (int t = t0 + 1; t < t1; ++t) {
            const float w = v[t];
            alone = alone || !(w == w);
            if (!(w < vb)) {
                best = t;
                vb = w;
            }
        }
#pragma unroll
        for (int off = 1; off < 64; off <<= 1) {  // lane l holds the runs l .. l + 2 off - 1
            const int ob = __shfl_down(best, off);
            const float ov = __shfl_down(vb, off);
            const bool oa = __shfl_down((int)alone, off) != 0, on = __shfl_down((int)any, off) != 0;
            if (lane + off < 64 && on && (oa || !(ov < vb))) {
                best = ob;
                vb = ov;
            }
            alone = alone || oa;
        }
        if (lane == 0) {
            part[0] = (uint32_t)best;
            *split_dim = best;
        }
    }
    for (int i = tid; i < 512; i += nt) hist[i] = 0u;
    __syncthreads();
    const int col = (int)part[0];
    for (uint32_t p = tid; p < cnt; p += nt) key[p] = float_order_key(x[(int64_t)perm[r.x + p] * ld + col]);
    __syncthreads();
    // both middle ranks, a byte per pass; waves 0 and 1 pick
    uint32_t pre0 = 0u, pre1 = 0u, rank0 = (cnt % 2 == 0) ? cnt / 2 - 1 : cnt / 2, rank1 = cnt / 2;
    for (int pass = 0; pass < 4; ++pass) {
        const int shift = 24 - 8 * pass;
        const uint32_t high = pass == 0 ? 0u : (0xFFFFFFFFu << (shift + 8));
        const bool same = pre0 == pre1;  // uniform: one histogram serves both
        for (uint32_t p = tid; p < cnt; p += nt) {
            const uint32_t k = key[p], byte = (k >> shift) & 255u;
            if ((k & high) == pre0) atomicAdd(&hist[byte], 1u);
            if (!same && (k & high) == pre1) atomicAdd(&hist[256 + byte], 1u);
        }
        __syncthreads();
        for (int w = wave; w < 2; w += nw) {
            const uint32_t *h = hist + (same ? 0 : 256 * w) + 4 * lane;
            const uint32_t c0 = h[0], c1 = h[1], c2 = h[2], tot = c0 + c1 + c2 + h[3], rank = w ? rank1 : rank0;
            uint32_t inc = tot;
#pragma unroll
            for (int off = 1; off < 64; off <<= 1) {
                const uint32_t v = __shfl_up(inc, off);
                if (lane >= off) inc += v;
            }
            uint32_t left = rank - (inc - tot);
            if (rank >= inc - tot && rank < inc) {  // one lane: every rank is below cnt
                uint32_t byte = 4u * (uint32_t)lane;
                if (left >= c0) {
                    left -= c0;
                    ++byte;
                    if (left >= c1) {
                        left -= c1;
                        ++byte;
                        if (left >= c2) {
                            left -= c2;
                            ++byte;
                        }
                    }
                }
                part[2 * w] = byte << shift;
                part[2 * w + 1] = left;
            }
        }
        __syncthreads();
        pre0 |= part[0];
        rank0 = part[1];
        pre1 |= part[2];
        rank1 = part[3];
        for (int i = tid; i < 512; i += nt) hist[i] = 0u;
        __syncthreads();
    }
    const float ma = float_from_order_key(pre0), mb = float_from_order_key(pre1), sum = ma + mb;
    const float med = (cnt % 2u == 0u) ? sum / 2.0f : ma;
    // left count, then the rows in order: each wave's share of a stretch of nt rows by its ballot
    uint32_t mine = 0;
    for (uint32_t p = tid; p < cnt; p += nt) mine += float_from_order_key(key[p]) <= med ? 1u : 0u;
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) mine += __shfl_xor(mine, off);
    if (lane == 0) part[wave] = mine;
    __syncthreads();
    uint32_t total = 0;
    for (int w = 0; w < nw; ++w) total += part[w];
    if (tid == 0) {
        *median = med;
        *nleft = total;
    }
    uint32_t before = 0;  // left rows of the stretches so far
    for (uint32_t base = 0; base < cnt; base += nt) {
        const uint32_t p = base + tid;
        const bool in = p < cnt, left = in && float_from_order_key(key[p]) <= med;
        const uint64_t m = __ballot(left);
        __syncthreads();  // (part has been read)
        if (lane == 0) part[wave] = (uint32_t)__popcll(m);
        __syncthreads();
        uint32_t mybefore = before + (uint32_t)__popcll(m & (((uint64_t)1 << lane) - 1));
        for (int w = 0; w < nw; ++w) {
            const uint32_t c = part[w];
            if (w < wave) mybefore += c;
            before += c;
        }
        if (in) perm_out[left ? r.x + mybefore : r.x + total + (p - mybefore)] = perm[r.x + p];
    }
    return total;
}

static __global__ void __launch_bounds__(1024) k_seg_split_wg(const uint32_t *__restrict__ perm,
                                                              const uint2 *__restrict__ seg_range,
                                                              const float *__restrict__ var, int dim, int stride,
                                                              const float *__restrict__ x, int64_t ld,
                                                              int *__restrict__ split_dim, float *__restrict__ median,
                                                              uint32_t *__restrict__ nleft, uint32_t *__restrict__ perm_out) {
    extern __shared__ uint32_t lds_split[];
    const int g = blockIdx.x;
    split_node(lds_split, lds_split + 512, lds_split + 576, perm, seg_range[g], var + (size_t)g * stride, dim, x, ld, split_dim + g,
               median + g, nleft + g, perm_out);
}

// ---- levels of short nodes, without the host between them ------------------------------------
// Where no node of a level is longer than var_tile_rows, the levels below it are built from tables on the device: the nodes of
// level d are the slots of a complete tree (children of slot g: 2 g and 2 g + 1 of the next table), a slot without a node
// is {0, 0}.  Every launch covers all slots of its level; the host reads the decisions of all levels at once and
// numbers the nodes.  (A level that waits for the host costs two copies, the wait and the time until its first kernel
// starts, 30 us on a level of 70-100, and its means were three launches where they are one or two.  Builds: 2,295 x 128, seven levels 398 -> 226 us,
// 4,157 x 100, ten 625 -> 361, 16,000 x 100, ten 871 -> 550, 100,000 x 128, ten 1268 -> 1088.)  The host knows no node's
// size here, only the longest one's above: what a launch is sized for is the balanced tree's, and a longer node
// (equal values all go left) takes more rounds of the same loops.  Where that would be many (kUneven), the split of the level
// above sets the level's word of stop: its kernels and those of the levels below return, and the host takes up there with
// the true length.  (A tree that ends early pays for the launches of its empty levels: thirteen levels of 2,000 rows of which three
// differ 170 -> 220 us, ten of 16,000 of which nine differ 573 -> 490.)
constexpr int kNodeLeaves = 16;  // leaves of 1024 rows of the longest node

// Rows lo .. hi - 1 (of cnt) of leaf l, by the midpoints of src/vector.rs's recursion.
__device__ __forceinline__ uint2 leaf_range(uint32_t cnt, int dep, uint32_t l) {
    uint32_t lo = 0, hi = cnt;
    for (int bit = dep - 1; bit >= 0; --bit) {
        const uint32_t mid = lo + (hi - lo) / 2;
        if ((l >> bit) & 1u)
            lo = mid;
        else
            hi = mid;
    }
    return make_uint2(lo, hi);
}

__device__ __forceinline__ int leaf_depth(uint32_t cnt) {
    int dep = 0;
    while (cnt > (1024u << dep)) ++dep;
    return dep;
}

// Sums of the leaves of a level's nodes, a workgroup per (node, one of every `per` leaves, tile of up to 32 components, as
// k_node_stats has them): leaf_sum[(node * kNodeLeaves + leaf) * dim + component].
template <int VEC, bool CHAIN>
static __global__ void __launch_bounds__(256) k_node_leafsum(const uint32_t *__restrict__ perm, const uint2 *__restrict__ range,
                                                             const uint32_t *__restrict__ stop, int slots, int per,
                                                             const float *__restrict__ x, int64_t ld, int dim, int width, int pieces,
                                                             float *__restrict__ leaf_sum) {
    extern __shared__ float4 lds_node[];
    const int g = blockIdx.x % (unsigned)slots, rest = blockIdx.x / (unsigned)slots, tile = rest / per;
    const int c0 = tile * width < dim - width ? tile * width : dim - width;
    const uint2 r = range[g];
    const uint32_t cnt = r.y - r.x;
    if (*stop) return;
    const int dep = leaf_depth(cnt);
    for (uint32_t l = (uint32_t)(rest % per); cnt && l < (1u << dep); l += (uint32_t)per) {
        const uint2 lr = leaf_range(cnt, dep, l);
        const float sum = tile_sum<256, VEC, false, CHAIN>(reinterpret_cast<float *>(lds_node), x + c0, ld, r.x + lr.x, r.x + lr.y, width, pieces,
                                                    [&](uint32_t p) { return perm[p]; });
        if ((int)threadIdx.x < width) leaf_sum[((size_t)g * kNodeLeaves + l) * dim + c0 + threadIdx.x] = sum;
        __syncthreads();  // (the stage has been read)
    }
}

// Means, and with var the sums of squared deviations, of a level's nodes: a workgroup per node and tile, as
// k_seg_variance_tile.  SUMS: the leaves are summed here, one after the other (nodes of up to 1024 rows have one); else from leaf_sum.
// NT threads: 64 for nodes of up to 256 rows, whose chunks of 128 members leave room for more workgroups (the last levels
// of 100,000 x 128, nodes of 195 and 98 rows: 23 -> 15 us each).
template <int VEC, bool SUMS, int NT, bool CHAIN>
static __global__ void __launch_bounds__(NT) k_node_stats(const uint32_t *__restrict__ perm, const uint2 *__restrict__ range,
                                                           const uint32_t *__restrict__ stop, int slots,
                                                           const float *__restrict__ x, int64_t ld, int dim, int width, int pieces,
                                                           const float *__restrict__ leaf_sum, float *__restrict__ means,
                                                           float *__restrict__ var) {
    extern __shared__ float4 lds_node[];
    __shared__ float leaf[kNodeLeaves][32];
    float *stage = reinterpret_cast<float *>(lds_node);
    const int g = blockIdx.x % (unsigned)slots, tile = blockIdx.x / (unsigned)slots, tid = threadIdx.x;
    const int c0 = tile * width < dim - width ? tile * width : dim - width;
    const uint2 r = range[g];
    const uint32_t cnt = r.y - r.x;
    if (*stop || cnt == 0) return;
    const int dep = leaf_depth(cnt);
    const uint32_t nl = 1u << dep;
    for (uint32_t l = 0; l < nl; ++l) {
        if constexpr (SUMS) {
            const uint2 lr = leaf_range(cnt, dep, l);
            const auto row = [&](uint32_t p) { return perm[p]; };
            const float sum = tile_sum<NT, VEC, false, CHAIN>(stage, x + c0, ld, r.x + lr.x, r.x + lr.y, width, pieces, row);
            if (tid < width) leaf[l][tid] = sum;
            __syncthreads();  // (the stage has been read)
        } else if (tid < width) {
            leaf[l][tid] = leaf_sum[((size_t)g * kNodeLeaves + l) * dim + c0 + tid];
        }
    }
    if (tid < width) {  // (a lane reads what it wrote itself)
        for (uint32_t h = 1; h < nl; h <<= 1)
            for (uint32_t q = 0; q < nl; q += 2 * h) leaf[q][tid] = leaf[q][tid] + leaf[q + h][tid];
        leaf[0][tid] = leaf[0][tid] / __uint2float_rn(cnt);
        means[(size_t)g * dim + c0 + tid] = leaf[0][tid];
    }
    if (!var || cnt < 2) return;
    __syncthreads();
    const auto row = [&](uint32_t p) { return perm[p]; };
    const float sum = tile_sum<NT, VEC, true, CHAIN>(stage, x + c0, ld, r.x, r.y, width, pieces, row, leaf[0]);
    if (tid < width) var[(size_t)g * dim + c0 + tid] = sum;
}

// k_seg_split_wg for the slots of a level; the children's positions go into the next level's table.  room: rows whose keys the
// workgroup's LDS holds; a longer node's keys lie in memory (keys, by position).  nleft stays 0 where nothing is split.
// most: rows of a child above which the next level stops (*stop: this level has).
static __global__ void __launch_bounds__(1024) k_node_split(const uint32_t *__restrict__ perm, const uint2 *__restrict__ range, uint32_t *stop,
                                                            uint32_t room, uint32_t most, const float *__restrict__ var, int dim, int stride,
                                                            const float *__restrict__ x, int64_t ld, uint32_t *__restrict__ keys,
                                                            int *__restrict__ split_dim, float *__restrict__ median,
                                                            uint32_t *__restrict__ nleft, uint32_t *__restrict__ perm_out,
                                                            uint2 *__restrict__ child) {
    extern __shared__ uint32_t lds_split[];
    uint32_t *hist = lds_split, *part = hist + 512;
    const int g = blockIdx.x;
    const uint2 r = range[g];
    const uint32_t cnt = r.y - r.x;
    if (*stop) {
        if (g == 0 && threadIdx.x == 0) stop[1] = 1u;
        return;
    }
    uint32_t nl = 0;
    const float *v = var + (size_t)g * stride;
    if (cnt >= 2 && cnt <= room)
        nl = split_node(hist, part, part + 64, perm, r, v, dim, x, ld, split_dim + g, median + g, nleft + g, perm_out);
    else if (cnt >= 2)
        nl = split_node(hist, part, keys + r.x, perm, r, v, dim, x, ld, split_dim + g, median + g, nleft + g, perm_out);
    if (threadIdx.x == 0) {
        const bool both = nl > 0 && nl < cnt;  // (no child holds all rows)
        if (cnt < 2) nleft[g] = 0u;
        if (both && (nl > cnt - nl ? nl : cnt - nl) > most) stop[1] = 1u;
        child[2 * g] = both ? make_uint2(r.x, r.x + nl) : make_uint2(0u, 0u);
        child[2 * g + 1] = both ? make_uint2(r.x + nl, r.y) : make_uint2(0u, 0u);
    }
}

// out[i][t] = means[idx[i]][t]: the means of the nodes that split, side by side
static __global__ void __launch_bounds__(256) k_gather_means(const float *__restrict__ means,
                                                             const int *__restrict__ idx, int ns, int dim,
                                                             float *__restrict__ out) {
    const int64_t e = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (e >= (int64_t)ns * dim) return;
    out[e] = means[(size_t)idx[e / dim] * dim + e % dim];
}

// ---- descent -------------------------------------------------------------------------------
template <int METRIC>
__device__ __forceinline__ float tsvq_dist(const float *__restrict__ xr, const float *__restrict__ c,
                                           int dim, float na, float nb) {
    float acc = 0.0f;
    if constexpr (METRIC == M_COS) {
        for (int t = 0; t < dim; ++t) {
            float p = xr[t] * c[t];
            acc = acc + p;
        }
        float den = na * nb;
        float q = acc / den;
        float d = 1.0f - q;
        return (na == 0.0f || nb == 0.0f) ? 1.0f : d;
    } else if constexpr (METRIC == M_L1) {
        for (int t = 0; t < dim; ++t) {
            float d = xr[t] - c[t];
            acc = acc + fabsf(d);
        }
        return acc;
    } else {
        for (int t = 0; t < dim; ++t) {
            float d = xr[t] - c[t];
            float p = d * d;
            acc = acc + p;
        }
        return METRIC == M_EUCLID ? sqrtf(acc) : acc;
    }
}

// One lane = one row; walks from the root, `<=` goes left (src/tsvq.rs:171), single children are
// followed unconditionally (177-178).  Both distances of a level are accumulated together.
template <int METRIC>
__global__ void __launch_bounds__(256) k_tsvq_descend(const float *__restrict__ x, int64_t n, int64_t ld,
                                                      int dim, const float *__restrict__ cen,
                                                      const float *__restrict__ cnorm,
                                                      const int *__restrict__ left,
                                                      const int *__restrict__ right,
                                                      int *__restrict__ leaf) {
    int64_t row = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (row >= n) return;
    const float *__restrict__ xr = x + row * ld;
    float na = 0.0f;
    if constexpr (METRIC == M_COS) {
        float sa = 0.0f;
        for (int t = 0; t < dim; ++t) {
            float p = xr[t] * xr[t];
            sa = sa + p;
        }
        na = sqrtf(sa);
    }
    int node = 0;
    for (;;) {
        int l = left[node], r = right[node];
        if (l >= 0 && r >= 0) {
            const float *__restrict__ cl = cen + (size_t)l * dim;
            const float *__restrict__ cr = cen + (size_t)r * dim;
            float al = 0.0f, ar = 0.0f;
            for (int t = 0; t < dim; ++t) {
                float xv = xr[t];
                if constexpr (METRIC == M_COS) {
                    float pl = xv * cl[t], pr = xv * cr[t];
                    al = al + pl;
                    ar = ar + pr;
                } else if constexpr (METRIC == M_L1) {
                    float dl = xv - cl[t], dr = xv - cr[t];
                    al = al + fabsf(dl);
                    ar = ar + fabsf(dr);
                } else {
                    float dl = xv - cl[t], dr = xv - cr[t];
                    float pl = dl * dl, pr = dr * dr;
                    al = al + pl;
                    ar = ar + pr;
                }
            }
            float dl, dr;
            if constexpr (METRIC == M_COS) {
                float nl = cnorm[l], nr = cnorm[r];
                float ql = al / (na * nl), qr = ar / (na * nr);
                dl = (na == 0.0f || nl == 0.0f) ? 1.0f : 1.0f - ql;
                dr = (na == 0.0f || nr == 0.0f) ? 1.0f : 1.0f - qr;
            } else if constexpr (METRIC == M_EUCLID) {
                dl = sqrtf(al);
                dr = sqrtf(ar);
            } else {
                dl = al;
                dr = ar;
            }
            node = (dl <= dr) ? l : r;
        } else if (l >= 0) {
            node = l;
        } else if (r >= 0) {
            node = r;
        } else {
            break;
        }
    }
    leaf[row] = node;
}

// The same walk with the row held in registers (DIM a multiple of 32 up to 128).  One wave = 64
// rows, eight waves per workgroup: the rows are read with whole-line loads through a small padded LDS tile, so every byte of
// the input is fetched once; the two child centroids of a lane's node are read 64 bytes at a
// time, the next piece in flight while the current one is accumulated.  The sums stay one
// sequential chain per (row, child), as in the reference.
template <int METRIC>
__device__ __forceinline__ void tsvq_step(float &al, float &ar, float xv, float cl, float cr) {
    if constexpr (METRIC == M_COS) {
        float pl = xv * cl, pr = xv * cr;
        al = al + pl;
        ar = ar + pr;
    } else if constexpr (METRIC == M_L1) {
        float dl = xv - cl, dr = xv - cr;
        al = al + fabsf(dl);
        ar = ar + fabsf(dr);
    } else {
        float dl = xv - cl, dr = xv - cr;
        float pl = dl * dl, pr = dr * dr;
        al = al + pl;
        ar = ar + pr;
    }
}

// The centroids of the first kTopNodes nodes (the upper levels of a tree numbered level by level)
// are staged in LDS: down there the lanes of a wave sit on a handful of nodes, and per-lane
// global reads of a few distinct lines cost the address unit as much as fully scattered ones.  Row
// stride DIM + 4: the 16-byte reads of up to 8 nodes at the same offset fall into different banks.
constexpr int kTopNodes = 255;  // levels 0-7 of a complete tree

template <int METRIC, int DIM>
__global__ void __launch_bounds__(512) k_tsvq_descend_reg(const float *__restrict__ x, int64_t n, int64_t ld,
                                                         const float *__restrict__ cen,
                                                         const float *__restrict__ cnorm,
                                                         const int *__restrict__ left,
                                                         const int *__restrict__ right, int n_nodes,
                                                         int *__restrict__ leaf) {
    constexpr int TS = DIM + 4;
    // The centroids of the first nodes are staged once per workgroup; the workgroup then walks over
    // batches of 8 x 64 rows (grid: one workgroup per compute unit), every lane fetching its own
    // row with 16-byte loads, all of them in flight together.
    constexpr int kTopFloats = kTopNodes * TS;
    __shared__ float lds[kTopFloats];
    __shared__ int lds_child[2 * kTopNodes];  // children of the staged nodes: the walk's dependent reads stay in LDS
    const int lane = threadIdx.x & 63;
    float *top = lds;
    const int ntop = n_nodes < kTopNodes ? n_nodes : kTopNodes;
    __shared__ float lds_cn[kTopNodes];  // their norms (cosine)
    for (int e = threadIdx.x; e < ntop; e += 512) {
        lds_child[2 * e] = left[e];
        lds_child[2 * e + 1] = right[e];
        if constexpr (METRIC == M_COS) lds_cn[e] = cnorm[e];
    }
    for (int e = threadIdx.x; e < ntop * (DIM / 4); e += 512) {
        const int nd = e / (DIM / 4), pc = e % (DIM / 4);
        *reinterpret_cast<float4 *>(&top[nd * TS + pc * 4]) =
            *reinterpret_cast<const float4 *>(cen + (size_t)nd * DIM + pc * 4);
    }
    __syncthreads();
    const int64_t nbatch = (n + 63) / 64;
    for (int64_t batch = (int64_t)blockIdx.x * 8 + (threadIdx.x >> 6); batch < nbatch; batch += (int64_t)gridDim.x * 8) {
    const int64_t row0 = batch * 64;  // one wave = 64 rows
    float xr[DIM];
    {
        const int64_t row = row0 + lane < n ? row0 + lane : n - 1;  // past the end: the last row, not stored
        const float4 *xp = reinterpret_cast<const float4 *>(x + row * ld);
#pragma unroll
        for (int q = 0; q < DIM / 4; ++q) {
            const float4 v = xp[q];
            xr[q * 4 + 0] = v.x;
            xr[q * 4 + 1] = v.y;
            xr[q * 4 + 2] = v.z;
            xr[q * 4 + 3] = v.w;
        }
    }
    float na = 0.0f;
    if constexpr (METRIC == M_COS) {
        float sa = 0.0f;
#pragma unroll
        for (int t = 0; t < DIM; ++t) {
            float p = xr[t] * xr[t];
            sa = sa + p;
        }
        na = sqrtf(sa);
    }
    int node = 0;
    bool active = row0 + lane < n;
    while (__any(active)) {
        int l = -1, r = -1;
        if (active) {
            if (node < ntop) {
                l = lds_child[2 * node];
                r = lds_child[2 * node + 1];
            } else {
                l = left[node];
                r = right[node];
            }
        }
        const bool both = l >= 0 && r >= 0;
        // every lane that compares two children finds them in LDS: the whole wave reads there
        if (!__any(both && (l >= ntop || r >= ntop))) {
            if (both) {
                const float *pl = &top[l * TS], *pr = &top[r * TS];
                float al = 0.0f, ar = 0.0f;
#pragma unroll
                for (int q = 0; q < DIM / 4; ++q) {
                    const float4 a = *reinterpret_cast<const float4 *>(pl + q * 4);
                    const float4 b = *reinterpret_cast<const float4 *>(pr + q * 4);
                    tsvq_step<METRIC>(al, ar, xr[q * 4 + 0], a.x, b.x);
                    tsvq_step<METRIC>(al, ar, xr[q * 4 + 1], a.y, b.y);
                    tsvq_step<METRIC>(al, ar, xr[q * 4 + 2], a.z, b.z);
                    tsvq_step<METRIC>(al, ar, xr[q * 4 + 3], a.w, b.w);
                }
                float dl, dr;
                if constexpr (METRIC == M_COS) {
                    float nl = lds_cn[l], nr = lds_cn[r];
                    float ql = al / (na * nl), qr = ar / (na * nr);
                    dl = (na == 0.0f || nl == 0.0f) ? 1.0f : 1.0f - ql;
                    dr = (na == 0.0f || nr == 0.0f) ? 1.0f : 1.0f - qr;
                } else if constexpr (METRIC == M_EUCLID) {
                    dl = sqrtf(al);
                    dr = sqrtf(ar);
                } else {
                    dl = al;
                    dr = ar;
                }
                node = (dl <= dr) ? l : r;
            } else if (l >= 0) {
                node = l;
            } else if (r >= 0) {
                node = r;
            } else {
                active = false;
            }
            continue;
        }
        if (both) {
            const float4 *pl = reinterpret_cast<const float4 *>(cen + (size_t)l * DIM);
            const float4 *pr = reinterpret_cast<const float4 *>(cen + (size_t)r * DIM);
            float al = 0.0f, ar = 0.0f;
            float4 bl[2][4], br[2][4];
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                bl[0][q] = pl[q];
                br[0][q] = pr[q];
            }
#pragma unroll
            for (int c = 0; c < DIM / 16; ++c) {
                if (c + 1 < DIM / 16) {
#pragma unroll
                    for (int q = 0; q < 4; ++q) {
                        bl[(c + 1) & 1][q] = pl[(c + 1) * 4 + q];
                        br[(c + 1) & 1][q] = pr[(c + 1) * 4 + q];
                    }
                }
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    const float4 a = bl[c & 1][q], b = br[c & 1][q];
                    tsvq_step<METRIC>(al, ar, xr[c * 16 + q * 4 + 0], a.x, b.x);
                    tsvq_step<METRIC>(al, ar, xr[c * 16 + q * 4 + 1], a.y, b.y);
                    tsvq_step<METRIC>(al, ar, xr[c * 16 + q * 4 + 2], a.z, b.z);
                    tsvq_step<METRIC>(al, ar, xr[c * 16 + q * 4 + 3], a.w, b.w);
                }
            }
            float dl, dr;
            if constexpr (METRIC == M_COS) {
                float nl = cnorm[l], nr = cnorm[r];
                float ql = al / (na * nl), qr = ar / (na * nr);
                dl = (na == 0.0f || nl == 0.0f) ? 1.0f : 1.0f - ql;
                dr = (na == 0.0f || nr == 0.0f) ? 1.0f : 1.0f - qr;
            } else if constexpr (METRIC == M_EUCLID) {
                dl = sqrtf(al);
                dr = sqrtf(ar);
            } else {
                dl = al;
                dr = ar;
            }
            node = (dl <= dr) ? l : r;
        } else if (l >= 0) {
            node = l;
        } else if (r >= 0) {
            node = r;
        } else {
            active = false;
        }
    }
    if (row0 + lane < n) leaf[row0 + lane] = node;
    }  // batches
}

// ---- descent decided by one inner product per node, exact where that cannot decide ---------------
// Cosine: the reference goes left iff dl <= dr with dl = 1 - (x.cl) / (|x| |cl|) (src/tsvq.rs:167-171,
// src/distances.rs:141-151), which in exact arithmetic is the sign of x.w, w = cl / |cl| - cr / |cr|.
// Squared Euclidean and Euclidean: the sign of x.w + b, w = 2 (cl - cr), b = |cr|^2 - |cl|^2.  So a
// node costs one vector of the table below instead of two centroids, and one chain of fused
// multiply-adds instead of two of rounded products.  The rounded sums of the reference can only
// differ from that sign when the value is small, and how small is bounded (u = 2^-24, D <= 128):
//   cosine   each of dl, dr is within 133.2 u of its exact value (129 u for the sequential sum of D
//            rounded products, relative to |x| |c|; 2 u for the product of the norms and the division;
//            2 u for 1 - q), the computed x.w within 260.1 u |x| of the exact one (4 u |x| from the
//            rounding of w, 256 u |x| from the sum): |x.w| > 600 u na decides, na the computed |x|.
//   L2       each of the sums within 131 u of its exact value, relatively; the roots of two sums that
//            differ by more than 6 u, relatively, differ after rounding; the computed x.w + b within
//            131 u S of the exact one, S = 4 |x|^2 + 2 (|cl|^2 + |cr|^2) >= both sums together:
//            |x.w + b| > 300 u (4 x2 + s) decides, x2 the computed |x|^2, s rounded up.
// Everything else — near ties, norms outside [1e-15, 1e15] (zero norms have their own rule in the
// reference, huge ones overflow), non-finite values (they fail the comparison) — is decided for that
// lane by the two sums in the reference's order, read from global memory.  Manhattan has no such form
// and keeps the two-centroid kernel.
// With D components the bounds are (4 D + 15) u and (2 D + 12) u; wider rows take margins that grow with them
// (600 u and 300 u at 128).
__host__ __device__ inline float descend_cos_margin(int dim) {
    return (float)(4 * (dim > 128 ? dim : 128) + 88) * 5.9604644775390625e-08f;
}
__host__ __device__ inline float descend_l2_margin(int dim) {
    return (float)(2 * (dim > 128 ? dim : 128) + 44) * 5.9604644775390625e-08f;
}

// Tables for the nodes below kTopNodes, one wave per node: w[node][DIM], and per node
//   cosine: sc[node] = descend_cos_margin, or +inf when a child's norm is outside [1e-15, 1e15]
//   L2:     sc[2 node] = b, sc[2 node + 1] = descend_l2_margin * s (+inf when s is not in [1e-30, 1e30])
// Nodes without two children get zeros and +inf (they are never consulted).
template <bool COS>
static __global__ void __launch_bounds__(64) k_tsvq_wtable(const float *__restrict__ cen,
                                                           const float *__restrict__ cnorm,
                                                           const int *__restrict__ left,
                                                           const int *__restrict__ right, int dim,
                                                           float *__restrict__ w, float *__restrict__ sc) {
    const int node = blockIdx.x, lane = threadIdx.x;
    const int l = left[node], r = right[node];
    const bool both = l >= 0 && r >= 0;
    const float inf = __builtin_inff();
    if (!both) {
        for (int t = lane; t < dim; t += 64) w[(size_t)node * dim + t] = 0.0f;
        if (lane == 0) {
            if (COS) {
                sc[node] = inf;
            } else {
                sc[2 * node] = 0.0f;
                sc[2 * node + 1] = inf;
            }
        }
        return;
    }
    const float *cl = cen + (size_t)l * dim, *cr = cen + (size_t)r * dim;
    if constexpr (COS) {
        const float nl = cnorm[l], nr = cnorm[r];
        for (int t = lane; t < dim; t += 64) {
            const float a = cl[t] / nl, b = cr[t] / nr;
            w[(size_t)node * dim + t] = a - b;
        }
        const bool ok = nl >= 1e-15f && nl <= 1e15f && nr >= 1e-15f && nr <= 1e15f;
        if (lane == 0) sc[node] = ok ? descend_cos_margin(dim) : inf;
    } else {
        double sl = 0.0, sr = 0.0;
        for (int t = lane; t < dim; t += 64) {
            const float a = cl[t], b = cr[t];
            w[(size_t)node * dim + t] = 2.0f * (a - b);
            sl += (double)a * (double)a;
            sr += (double)b * (double)b;
        }
#pragma unroll
        for (int off = 32; off > 0; off >>= 1) {
            sl += __shfl_xor(sl, off);
            sr += __shfl_xor(sr, off);
        }
        if (lane == 0) {
            const double s = 2.0 * (sl + sr);
            const bool ok = s >= 1e-30 && s <= 1e30;  // false for NaN
            sc[2 * node] = (float)(sr - sl);
            sc[2 * node + 1] = ok ? (float)(s * 1.000001) * descend_l2_margin(dim) : inf;
        }
    }
}

// The walk of k_tsvq_descend_reg with the decision above: the table of the first kTopNodes nodes
// in LDS (same layout and stride), the row in registers.  METRIC: M_SQ, M_EUCLID or M_COS.
template <int METRIC, int DIM>
__global__ void __launch_bounds__(512) k_tsvq_descend_w(const float *__restrict__ x, int64_t n, int64_t ld,
                                                       const float *__restrict__ cen,
                                                       const float *__restrict__ cnorm,
                                                       const int *__restrict__ left,
                                                       const int *__restrict__ right, int n_nodes,
                                                       const float *__restrict__ wtab,
                                                       const float *__restrict__ sctab, int *__restrict__ leaf) {
    constexpr int TS = DIM + 4;
    constexpr bool COS = METRIC == M_COS;
    __shared__ float top[kTopNodes * TS];
    __shared__ int lds_child[2 * kTopNodes];
    __shared__ float lds_sc[2 * kTopNodes];
    const int lane = threadIdx.x & 63;
    const int ntop = n_nodes < kTopNodes ? n_nodes : kTopNodes;
    for (int e = threadIdx.x; e < ntop; e += 512) {
        lds_child[2 * e] = left[e];
        lds_child[2 * e + 1] = right[e];
        if constexpr (COS) {
            lds_sc[e] = sctab[e];
        } else {
            lds_sc[2 * e] = sctab[2 * e];
            lds_sc[2 * e + 1] = sctab[2 * e + 1];
        }
    }
    for (int e = threadIdx.x; e < ntop * (DIM / 4); e += 512) {
        const int nd = e / (DIM / 4), pc = e % (DIM / 4);
        *reinterpret_cast<float4 *>(&top[nd * TS + pc * 4]) =
            *reinterpret_cast<const float4 *>(wtab + (size_t)nd * DIM + pc * 4);
    }
    __syncthreads();
    const int64_t nbatch = (n + 63) / 64;
    for (int64_t batch = (int64_t)blockIdx.x * 8 + (threadIdx.x >> 6); batch < nbatch; batch += (int64_t)gridDim.x * 8) {
        const int64_t row0 = batch * 64;  // one wave = 64 rows
        float xr[DIM];
        {
            const int64_t row = row0 + lane < n ? row0 + lane : n - 1;  // past the end: the last row, not stored
            const float4 *xp = reinterpret_cast<const float4 *>(x + row * ld);
#pragma unroll
            for (int q = 0; q < DIM / 4; ++q) {
                const float4 v = xp[q];
                xr[q * 4 + 0] = v.x;
                xr[q * 4 + 1] = v.y;
                xr[q * 4 + 2] = v.z;
                xr[q * 4 + 3] = v.w;
            }
        }
        // |x|^2 in the reference's order (the exact step's cosine needs it so; the margins take it as it is)
        float sa = 0.0f;
#pragma unroll
        for (int t = 0; t < DIM; ++t) {
            float p = xr[t] * xr[t];
            sa = sa + p;
        }
        const float na = sqrtf(sa);
        // the row's own share of the margin; a row whose norm is out of range (or not finite) never
        // passes the test: +inf
        const float inf = __builtin_inff();
        float mrow;
        if constexpr (COS)
            mrow = (na >= 1e-15f && na <= 1e15f) ? na : inf;
        else
            mrow = (sa <= 1e30f) ? 4.0f * descend_l2_margin(DIM) * sa : inf;  // false for NaN
        int node = 0;
        bool active = row0 + lane < n;
        while (__any(active)) {
            int l = -1, r = -1;
            if (active) {
                if (node < ntop) {
                    l = lds_child[2 * node];
                    r = lds_child[2 * node + 1];
                } else {
                    l = left[node];
                    r = right[node];
                }
            }
            const bool both = l >= 0 && r >= 0;
            bool undecided = both;
            if (both && node < ntop) {
                const float *pw = &top[node * TS];
                float f0 = 0.0f, f1 = 0.0f, f2 = 0.0f, f3 = 0.0f;
#pragma unroll
                for (int q = 0; q < DIM / 4; ++q) {
                    const float4 a = *reinterpret_cast<const float4 *>(pw + q * 4);
                    f0 = __builtin_fmaf(xr[q * 4 + 0], a.x, f0);
                    f1 = __builtin_fmaf(xr[q * 4 + 1], a.y, f1);
                    f2 = __builtin_fmaf(xr[q * 4 + 2], a.z, f2);
                    f3 = __builtin_fmaf(xr[q * 4 + 3], a.w, f3);
                }
                float f = (f0 + f1) + (f2 + f3);
                float theta;
                if constexpr (COS) {
                    theta = lds_sc[node] * mrow;
                } else {
                    f += lds_sc[2 * node];
                    theta = lds_sc[2 * node + 1] + mrow;
                }
                // (inf * 0 and inf - inf give NaN, which fails both tests)
                if (f > theta) {
                    node = l;
                    undecided = false;
                } else if (f < -theta) {
                    node = r;
                    undecided = false;
                }
            } else if (!both) {
                if (l >= 0)
                    node = l;
                else if (r >= 0)
                    node = r;
                else
                    active = false;
            }
            if (__any(undecided)) {
                if (undecided) {
                    // the two sums in the reference's order (src/tsvq.rs:167-171), from global memory
                    const float4 *pl = reinterpret_cast<const float4 *>(cen + (size_t)l * DIM);
                    const float4 *pr = reinterpret_cast<const float4 *>(cen + (size_t)r * DIM);
                    float al = 0.0f, ar = 0.0f;
#pragma unroll
                    for (int q = 0; q < DIM / 4; ++q) {
                        const float4 a = pl[q], b = pr[q];
                        tsvq_step<METRIC>(al, ar, xr[q * 4 + 0], a.x, b.x);
                        tsvq_step<METRIC>(al, ar, xr[q * 4 + 1], a.y, b.y);
                        tsvq_step<METRIC>(al, ar, xr[q * 4 + 2], a.z, b.z);
                        tsvq_step<METRIC>(al, ar, xr[q * 4 + 3], a.w, b.w);
                    }
                    float dl, dr;
                    if constexpr (COS) {
                        float nl = cnorm[l], nr = cnorm[r];
                        float ql = al / (na * nl), qr = ar / (na * nr);
                        dl = (na == 0.0f || nl == 0.0f) ? 1.0f : 1.0f - ql;
                        dr = (na == 0.0f || nr == 0.0f) ? 1.0f : 1.0f - qr;
                    } else if constexpr (METRIC == M_EUCLID) {
                        dl = sqrtf(al);
                        dr = sqrtf(ar);
                    } else {
                        dl = al;
                        dr = ar;
                    }
                    node = (dl <= dr) ? l : r;
                }
            }
        }
        if (row0 + lane < n) leaf[row0 + lane] = node;
    }  // batches
}

// The walk for every width up to 256 and rows of any alignment: four lanes per row, lane q with the pieces 4 p + q of
// four components (zeros behind the last one), so that a row's four lanes read 64 consecutive bytes and a wave holds
// 16 rows in NP * 4 registers per lane.  The inner product decides as above where the node has a table (below ntab; the
// first ntop of it in LDS).  Else both children's sums are made from memory, each lane its pieces with fused
// multiply-adds, and their difference decides where it exceeds the bounds on both roundings:
//   L2         |ar - al| > (2 D + 13) u (al + ar), al + ar >= 1e-30 (no square has lost bits below the smallest number)
//   Manhattan  |ar - al| > (2 D + 2) u (al + ar)
//   cosine     |pl / |cl| - pr / |cr|| > (4 D + 17) u |x|, norms as above
// (the margins of descend_l2_margin and descend_cos_margin cover them; those of L2 are the distances' share and not
// the vectors': rows far from the origin, as uniform ones are, 16 times closer at 248 components).  What that cannot
// decide takes the two sums in the reference's order, lane 0 the left one, lane 1 the right one.  Manhattan has no
// table: its LDS holds the first ntop centroids.
// The nodes' stride of an odd number of 64-byte pieces spreads the rows of a wave over the banks.
typedef float quad_piece __attribute__((ext_vector_type(4), aligned(4)));

__host__ __device__ constexpr int quad_stride(int np) { return 16 * (np | 1); }

// Workgroups of 512 threads per compute unit: what the registers allow.
__host__ __device__ constexpr int quad_per_cu(int np) { return np <= 2 ? 3 : np <= 7 ? 2 : 1; }

__device__ __forceinline__ quad_piece quad_load(const float *__restrict__ p, int at, int dim) {
    quad_piece v = {0.0f, 0.0f, 0.0f, 0.0f};
    if (at + 4 <= dim) {
        v = *reinterpret_cast<const quad_piece *>(p + at);
    } else {
        if (at < dim) v.x = p[at];
        if (at + 1 < dim) v.y = p[at + 1];
        if (at + 2 < dim) v.z = p[at + 2];
    }
    return v;
}

// What lane LANE of a row's four holds.
template <int LANE>
__device__ __forceinline__ float quad_from(float v) {
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), LANE * 0x55, 0xf, 0xf, false));
}

// The sum over a row's four lanes, the same bits in each of them.
__device__ __forceinline__ float quad_sum(float v) {
    v += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0xB1, 0xf, 0xf, false));  // lanes 1 0 3 2
    v += __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x4E, 0xf, 0xf, false));  // lanes 2 3 0 1
    return v;
}

// Both children's sums over a lane's pieces, in an order of their own.
template <int METRIC, int NP, typename Load>
__device__ __forceinline__ void quad_pair(const quad_piece (&xr)[NP], float &sl, float &sr, Load load) {
    float al[2] = {0.0f, 0.0f}, ar[2] = {0.0f, 0.0f};
#pragma unroll
    for (int p = 0; p < NP; ++p) {
        quad_piece a, b;
        load(p, a, b);
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const float xv = xr[p][e];
            if constexpr (METRIC == M_COS) {
                al[e & 1] = __builtin_fmaf(xv, a[e], al[e & 1]);
                ar[e & 1] = __builtin_fmaf(xv, b[e], ar[e & 1]);
            } else if constexpr (METRIC == M_L1) {
                al[e & 1] += fabsf(xv - a[e]);
                ar[e & 1] += fabsf(xv - b[e]);
            } else {
                const float dl = xv - a[e], dr = xv - b[e];
                al[e & 1] = __builtin_fmaf(dl, dl, al[e & 1]);
                ar[e & 1] = __builtin_fmaf(dr, dr, ar[e & 1]);
            }
        }
    }
    sl = quad_sum(al[0] + al[1]);
    sr = quad_sum(ar[0] + ar[1]);
}

// tab: the table of k_tsvq_wtable with sctab, of ntab nodes, or the centroids themselves (Manhattan); ntop: the nodes of it in
// LDS.  OUT: the leaves' centroids into out16 as well, for a few rows: an instance of its own, as the common one has no registers for the loads of
// R rows (a row's load behind the store of the one before was 2 to 4 us of a call; 16 rows' loads are 1 us faster than four for 16 rows
// and more, and as much slower for one to three; above 208 components they spill).
template <int METRIC, int NP, bool OUT>
__global__ void __launch_bounds__(512, OUT ? 2 : 2 * quad_per_cu(NP)) k_tsvq_descend_quad(const float *__restrict__ x, int64_t n, int64_t ld, int dim,
                                                           const float *__restrict__ cen,
                                                           const float *__restrict__ cnorm,
                                                           const int *__restrict__ left,
                                                           const int *__restrict__ right,
                                                           const float *__restrict__ tab,
                                                           const float *__restrict__ sctab, int ntop, int ntab,
                                                           int *__restrict__ leaf, uint16_t *__restrict__ out16) {
    constexpr int S = quad_stride(NP), R = 4;
    constexpr bool COS = METRIC == M_COS, L1 = METRIC == M_L1;
    extern __shared__ float4 lds_quad[];  // [ntop][S] the nodes, [2 ntop] their children, [2 ntop] their scalars
    float *top = reinterpret_cast<float *>(lds_quad);
    int *child = reinterpret_cast<int *>(top + (size_t)ntop * S);
    float *sc = reinterpret_cast<float *>(child + 2 * ntop);
    const float inf = __builtin_inff();
    for (int e = threadIdx.x; e < ntop; e += blockDim.x) {
        child[2 * e] = left[e];
        child[2 * e + 1] = right[e];
        if constexpr (COS) {
            sc[e] = sctab[e];
        } else if constexpr (!L1) {
            sc[2 * e] = sctab[2 * e];
            sc[2 * e + 1] = sctab[2 * e + 1];
        }
    }
    for (int e = threadIdx.x; e < ntop * NP * 4; e += blockDim.x) {
        const int nd = e / (NP * 4), pc = e % (NP * 4);
        *reinterpret_cast<float4 *>(&top[nd * S + pc * 4]) =
            __builtin_bit_cast(float4, quad_load(tab + (size_t)nd * dim, pc * 4, dim));
    }
    __syncthreads();
    const int q = threadIdx.x & 3, waves = blockDim.x >> 6;
    const float l2m = descend_l2_margin(dim), cosm = descend_cos_margin(dim);
    const int64_t nbatch = (n + 15) / 16;
    for (int64_t batch = (int64_t)blockIdx.x * waves + (threadIdx.x >> 6); batch < nbatch; batch += (int64_t)gridDim.x * waves) {
        const int64_t row = batch * 16 + ((threadIdx.x & 63) >> 2);
        const float *__restrict__ xp = x + (row < n ? row : n - 1) * ld;  // past the end: the last row, not stored
        quad_piece xr[NP];
#pragma unroll
        for (int p = 0; p < NP; ++p) xr[p] = quad_load(xp, (p * 4 + q) * 4, dim);
        float mrow = 0.0f;  // the row's own share of the margin, +inf where its norm is out of range or not finite
        if constexpr (!L1) {
            float s0 = 0.0f, s1 = 0.0f;
#pragma unroll
            for (int p = 0; p < NP; ++p) {
                s0 = __builtin_fmaf(xr[p][0], xr[p][0], s0);
                s1 = __builtin_fmaf(xr[p][1], xr[p][1], s1);
                s0 = __builtin_fmaf(xr[p][2], xr[p][2], s0);
                s1 = __builtin_fmaf(xr[p][3], xr[p][3], s1);
            }
            const float sa = quad_sum(s0 + s1), na = sqrtf(sa);
            if constexpr (COS)
                mrow = (na >= 1e-15f && na <= 1e15f) ? na : inf;
            else
                mrow = (sa <= 1e30f) ? 4.0f * l2m * sa : inf;  // false for NaN
        }
        int node = 0;
        bool active = row < n;
        while (__any(active)) {
            int l = -1, r = -1;
            if (active) {
                if (node < ntop) {
                    l = child[2 * node];
                    r = child[2 * node + 1];
                } else {
                    l = left[node];
                    r = right[node];
                }
            }
            if (l >= 0 && r >= 0) {  // (the four lanes of a row agree here and below)
                float f = 0.0f, theta = inf;
                if (!L1 && node < ntab) {
                    float f0 = 0.0f, f1 = 0.0f, f2 = 0.0f, f3 = 0.0f;
                    auto dot = [&](auto load) {
#pragma unroll
                        for (int p = 0; p < NP; ++p) {
                            const quad_piece a = load(p);
                            f0 = __builtin_fmaf(xr[p][0], a[0], f0);
                            f1 = __builtin_fmaf(xr[p][1], a[1], f1);
                            f2 = __builtin_fmaf(xr[p][2], a[2], f2);
                            f3 = __builtin_fmaf(xr[p][3], a[3], f3);
                        }
                    };
                    if (node < ntop) {
                        const float *pw = &top[node * S + q * 4];
                        dot([&](int p) { return __builtin_bit_cast(quad_piece, *reinterpret_cast<const float4 *>(pw + p * 16)); });
                    } else {
                        const float *pw = tab + (size_t)node * dim;
                        dot([&](int p) { return quad_load(pw, (p * 4 + q) * 4, dim); });
                    }
                    const float *sn = node < ntop ? sc : sctab;
                    f = quad_sum((f0 + f1) + (f2 + f3));
                    if constexpr (COS) {
                        theta = sn[node] * mrow;
                    } else {
                        f += sn[2 * node];
                        theta = sn[2 * node + 1] + mrow;
                    }
                }
                if (!(fabsf(f) > theta)) {  // (also for NaN)
                    float sl, sr;
                    if (L1 && l < ntop && r < ntop) {
                        const float *pl = &top[l * S + q * 4], *pr = &top[r * S + q * 4];
                        quad_pair<METRIC, NP>(xr, sl, sr, [&](int p, quad_piece &a, quad_piece &b) {
                            a = __builtin_bit_cast(quad_piece, *reinterpret_cast<const float4 *>(pl + p * 16));
                            b = __builtin_bit_cast(quad_piece, *reinterpret_cast<const float4 *>(pr + p * 16));
                        });
                    } else {
                        const float *pl = cen + (size_t)l * dim, *pr = cen + (size_t)r * dim;
                        quad_pair<METRIC, NP>(xr, sl, sr, [&](int p, quad_piece &a, quad_piece &b) {
                            a = quad_load(pl, (p * 4 + q) * 4, dim);
                            b = quad_load(pr, (p * 4 + q) * 4, dim);
                        });
                    }
                    if constexpr (COS) {
                        const float nl = cnorm[l], nr = cnorm[r];
                        const bool ok = nl >= 1e-15f && nl <= 1e15f && nr >= 1e-15f && nr <= 1e15f;
                        f = sl / nl - sr / nr;
                        theta = ok ? cosm * mrow : inf;
                    } else {
                        f = sr - sl;
                        theta = (L1 || sl + sr >= 1e-30f) ? l2m * (sl + sr) : inf;
                    }
                }
                if (f > theta) {  // (NaN fails both tests)
                    node = l;
                } else if (f < -theta) {
                    node = r;
                } else {
                    // the two sums in the reference's order (src/tsvq.rs:167-171)
                    const float *__restrict__ c = cen + (size_t)((q & 1) ? r : l) * dim;
                    float d = 0.0f, sa = 0.0f;
#pragma unroll 8
                    for (int t = 0; t < dim; ++t) {
                        const float xv = xp[t];
                        wide_step<METRIC>(d, xv, c[t]);
                        if constexpr (COS) {
                            const float xx = xv * xv;
                            sa = sa + xx;
                        }
                    }
                    if constexpr (COS) {
                        const float na = sqrtf(sa), nc = cnorm[(q & 1) ? r : l];
                        const float quot = d / (na * nc);
                        d = (na == 0.0f || nc == 0.0f) ? 1.0f : 1.0f - quot;
                    }
                    if constexpr (METRIC == M_EUCLID) d = sqrtf(d);
                    const float dl = quad_from<0>(d), dr = quad_from<1>(d);
                    node = dl <= dr ? l : r;
                }
            } else if (l >= 0) {
                node = l;
            } else if (r >= 0) {
                node = r;
            } else {
                active = false;
            }
        }
        if (q == 0 && row < n) leaf[row] = node;
        if constexpr (OUT)  // a row at a time by the whole wave: runs of 128 bytes, also into host memory; the loads of R rows in flight
            for (int i0 = 0; i0 < 16 && batch * 16 + i0 < n; i0 += R) {
                const float *c[R];
#pragma unroll
                for (int i = 0; i < R; ++i) c[i] = cen + (size_t)__builtin_amdgcn_readlane(node, 4 * (i0 + i)) * dim;
                for (int t = threadIdx.x & 63; t < dim; t += 64) {
                    float v[R];
#pragma unroll
                    for (int i = 0; i < R; ++i) v[i] = c[i][t];
#pragma unroll
                    for (int i = 0; i < R; ++i)
                        if (batch * 16 + i0 + i < n) out16[(batch * 16 + i0 + i) * dim + t] = __half_as_ushort(__float2half_rn(v[i]));
                }
            }
    }  // batches
}

// TSVQNode::quantize_with_distance (src/tsvq.rs:162-181) for a few rows: one wave per row, which brings
// both children's centroids of a node into LDS with whole-line loads; lane 0 adds up the left distance
// and lane 1 the right one, each in the reference's order.  out16 (nullable): the leaf's centroid.
// (For widths beyond k_tsvq_descend_quad, and where few levels are over before that kernel's table is read.)
template <int METRIC>
__global__ void __launch_bounds__(64) k_tsvq_few(const float *__restrict__ x, int64_t ld, int dim,
                                                 const float *__restrict__ cen, const float *__restrict__ cnorm,
                                                 const int *__restrict__ left, const int *__restrict__ right,
                                                 int *__restrict__ leaf, uint16_t *__restrict__ out16) {
    extern __shared__ float lds_few[];  // the row, the left centroid, the right one: rows of dim + 1
    const int lane = threadIdx.x;
    const int64_t row = blockIdx.x;
    const int stride = dim + 1;
    float *xs = lds_few, *cs = lds_few + stride;
    for (int t = lane; t < dim; t += 64) xs[t] = x[row * ld + t];
    __syncthreads();
    float na = 0.0f;
    if constexpr (METRIC == M_COS) {
        float sa = 0.0f;
        for (int t = 0; t < dim; ++t) {
            const float p = xs[t] * xs[t];
            sa = sa + p;
        }
        na = sqrtf(sa);
    }
    int node = 0;
    for (;;) {
        const int l = left[node], r = right[node];
        if (l < 0 && r < 0) break;
        if (l < 0 || r < 0) {
            node = l >= 0 ? l : r;
            continue;
        }
#pragma unroll 2
        for (int t = lane; t < dim; t += 64) {
            cs[t] = cen[(size_t)l * dim + t];
            cs[stride + t] = cen[(size_t)r * dim + t];
        }
        const float nc = METRIC == M_COS ? cnorm[lane == 0 ? l : r] : 0.0f;
        __syncthreads();
        const float *c = cs + (lane & 1) * stride;  // (the other lanes repeat these two sums)
        float acc = 0.0f;
#pragma unroll 8
        for (int t = 0; t < dim; ++t) wide_step<METRIC>(acc, xs[t], c[t]);
        float d = acc;
        if constexpr (METRIC == M_COS) {
            const float q = acc / (na * nc);
            d = (na == 0.0f || nc == 0.0f) ? 1.0f : 1.0f - q;
        }
        if constexpr (METRIC == M_EUCLID) d = sqrtf(d);
        const float dl = __shfl(d, 0), dr = __shfl(d, 1);
        node = dl <= dr ? l : r;
        __syncthreads();
    }
    if (lane == 0) leaf[row] = node;
    if (out16)
        for (int t = lane; t < dim; t += 64) out16[row * dim + t] = __half_as_ushort(__float2half_rn(cen[(size_t)node * dim + t]));
}

}  // namespace vq

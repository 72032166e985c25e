// Centroid update of the LBG loop (src/utils.rs:83-102) as a deterministic ordered sum.
//
// The reference gathers the members of every cluster in row order and calls mean_vector
// (src/vector.rs:282-318).  Order of the f32 additions, per cluster:
//   1..1024 members ("small"): one sequential sum in row order from 0.0 — the reference's own,
//       deterministic order.  The rows of the small clusters are grouped by code with a STABLE
//       counting sort (per-part histograms -> exclusive scans -> ballot-ranked scatter of row
//       ids) and every cluster's list is walked by one lane per component.
//   more than 1024 ("large"): the reference switches to a Rayon reduce whose tree depends on
//       work stealing and cannot be reproduced even by itself.  Here the order is fixed as:
//       the rows are cut into parts of 4096 consecutive rows; inside a part the cluster's
//       members are added in row order from 0.0; the per-part sums are added in part order
//       from 0.0.  For 32-byte sub-vectors this is one streaming pass over the rows
//       (k_lbg_stream8) with the accumulators in LDS; other shapes take per-part leaves
//       through the gather path.
// No floating-point atomics anywhere; integer LDS atomics only for the histograms.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "assign_mfma.hpp"
#include "member_tile.hpp"

namespace vq {

constexpr int kPartRows = 4096;      // rows per part (histogram block and summation part)
constexpr int kScanSeg = 32;         // parts per scan segment
constexpr int kMaxK = 256;           // codes are uint8
constexpr int kSeqMax = 1024;        // PARALLEL_THRESHOLD, src/vector.rs:16

struct LbgState {
    // per column block s
    int *changed;          // m
    int *done;             // m   of this iteration
    int *done_next = nullptr;  // m   of the next one: written with the plan where no later kernel controls the loop, else null
    int *iters;            // m
    int *used;             // m   re-seed entries consumed so far
    int *ubase;            // m   value of used[s] at the start of the current update
    int *nleaves;          // m
    int *nsmall;           // m   clusters with 1..1024 members
    int *err;              // 1   set to 1 when a re-seed stream runs out
    // per (s, j)
    uint32_t *count;       // m*256
    uint32_t *start;       // m*256 first position of cluster j in perm[s]
    uint32_t *leaf_start;  // m*256
    uint32_t *empty_rank;  // m*256 rank of an empty cluster among the empty clusters of s
    // bulk
    uint32_t *hist;        // m*nparts*256 (histogram, then exclusive prefix over parts)
    uint32_t *seg;         // m*nseg*256 (per-segment sums, then exclusive prefix over segments)
    uint32_t *perm;        // m*n  row ids grouped by code, row order inside a group
    uint2 *leaf_desc;      // m*leaf_cap  [lo, hi) positions in perm[s]
    float *leaf_sum;       // m*leaf_cap*sd
    float *part_sum;       // m*nparts*256*8 per-part sums of the streaming kernel, or null
    uint8_t *codes;        // m*n  (column-block major)
    int nparts;
    int nseg;
    int leaf_cap;
    int stream;            // 1: the large clusters are summed by k_lbg_stream8 / k_lbg_combine8
    // wide column blocks (k_lbg_leafsum_wide): the leaves {lo, hi, leaf} in the order in which they are summed, else
    // null: small clusters, then the large clusters' leaves part by part, long ones left out (leaf = kNoLeaf)
    uint4 *order = nullptr;       // m*leaf_cap
    uint4 *longs = nullptr;       // m*2*long_cap: leaves of kVeryLong members or more, leaves of kLong or more
    uint32_t *place = nullptr;    // m*256 rank of a cluster among the small or among the large ones
    int *nlong = nullptr;         // m*2
    int long_cap = 0;
};
constexpr uint32_t kNoLeaf = 0xffffffffu;
constexpr uint32_t kLong = 128, kVeryLong = 512;  // members

__device__ __forceinline__ int long_class(uint32_t len) { return len >= kVeryLong ? 0 : len >= kLong ? 1 : 2; }

// The short kernels of the gather path run beside the streaming kernel, whose waves keep the
// vector ALU busy: their waves are given the higher issue priority, or they would wait for it.
__device__ __forceinline__ void side_chain_priority() { __builtin_amdgcn_s_setprio(3); }

static __global__ void k_lbg_init(LbgState st, int m) {
    int s = blockIdx.x * blockDim.x + threadIdx.x;
    if (s < m) {
        st.changed[s] = 0;
        st.done[s] = 0;
        if (st.done_next) st.done_next[s] = 0;
        st.iters[s] = 0;
        st.used[s] = 0;
        st.ubase[s] = 0;
        st.nleaves[s] = 0;
        st.nsmall[s] = 0;
    }
    if (s == 0) st.err[0] = 0;
}

// codebook[s][j][t] = x[idx[s][j]][s*sd + t]     (src/utils.rs:54)
static __global__ void k_gather_rows(const float *__restrict__ x, int64_t ld, int m, int k, int sd,
                              const uint32_t *__restrict__ idx, float *__restrict__ cb) {
    int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    int64_t total = (int64_t)m * k * sd;
    if (i >= total) return;
    int t = (int)(i % sd);
    int64_t sj = i / sd;
    int s = (int)(sj / k);
    cb[i] = x[(int64_t)idx[sj] * ld + (int64_t)s * sd + t];
}

// The same from a residual whose update is still pending (one column block):
// codebook[j][t] = x[idx[j]][t] - pend_cb[pend_codes[idx[j]]][t], the row as the update will leave it.
static __global__ void k_gather_rows_pend(const float *__restrict__ x, int64_t ld, int k, int sd,
                                          const uint32_t *__restrict__ idx, float *__restrict__ cb,
                                          const float *__restrict__ pend_cb, const uint8_t *__restrict__ pend_codes) {
    int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= (int64_t)k * sd) return;
    const int t = (int)(i % sd);
    const uint32_t row = idx[i / sd];
    cb[i] = x[(int64_t)row * ld + t] - pend_cb[(size_t)pend_codes[row] * sd + t];
}

// One wave per (part, column block): histogram of the codes of kPartRows rows.
static __global__ void __launch_bounds__(64) k_lbg_hist(LbgState st, int64_t n) {
    side_chain_priority();
    const int s = blockIdx.y, b = blockIdx.x;
    if (st.done[s]) return;
    __shared__ uint32_t cnt[kMaxK];
    for (int j = threadIdx.x; j < kMaxK; j += 64) cnt[j] = 0;
    __syncthreads();
    const uint8_t *codes = st.codes + (size_t)s * n;
    int64_t lo = (int64_t)b * kPartRows;
    int64_t hi = lo + kPartRows < n ? lo + kPartRows : n;
    if (hi - lo == kPartRows && ((uintptr_t)(codes + lo) & 15) == 0) {
        // a full part: every lane takes 64 consecutive codes with four loads in flight together
        // (a histogram does not care which lane counts which row)
        const uint4 *cp = reinterpret_cast<const uint4 *>(codes + lo) + threadIdx.x * 4;
        uint4 v[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) v[u] = cp[u];
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            const uint32_t w[4] = {v[u].x, v[u].y, v[u].z, v[u].w};
#pragma unroll
            for (int q = 0; q < 4; ++q)
#pragma unroll
                for (int sh = 0; sh < 32; sh += 8) atomicAdd(&cnt[(w[q] >> sh) & 255u], 1u);
        }
    } else {
        for (int64_t i = lo + threadIdx.x; i < hi; i += 64) atomicAdd(&cnt[codes[i]], 1u);
    }
    __syncthreads();
    uint32_t *h = st.hist + ((size_t)s * st.nparts + b) * kMaxK;
    for (int j = threadIdx.x; j < kMaxK; j += 64) h[j] = cnt[j];
}

// The same by four waves with a histogram each, where no streaming kernel runs beside it (12 -> 6 us at 2 to 47 parts: the
// time is a wave's chain of LDS additions, and of few parts no other wave hides it).
static __global__ void __launch_bounds__(256) k_lbg_hist_wg(LbgState st, int64_t n) {
    const int s = blockIdx.y, b = blockIdx.x, w = threadIdx.x >> 6;
    if (st.done[s]) return;
    __shared__ uint32_t cnt[4][kMaxK];
    for (int j = threadIdx.x; j < 4 * kMaxK; j += 256) (&cnt[0][0])[j] = 0;
    __syncthreads();
    const uint8_t *codes = st.codes + (size_t)s * n;
    const int64_t lo = (int64_t)b * kPartRows;
    const int64_t hi = lo + kPartRows < n ? lo + kPartRows : n;
    if (hi - lo == kPartRows && ((uintptr_t)(codes + lo) & 15) == 0) {
        const uint4 v = reinterpret_cast<const uint4 *>(codes + lo)[threadIdx.x];
        const uint32_t q[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
        for (int u = 0; u < 4; ++u)
#pragma unroll
            for (int sh = 0; sh < 32; sh += 8) atomicAdd(&cnt[w][(q[u] >> sh) & 255u], 1u);
    } else {
        for (int64_t i = lo + threadIdx.x; i < hi; i += 256) atomicAdd(&cnt[w][codes[i]], 1u);
    }
    __syncthreads();
    const int j = threadIdx.x;
    st.hist[((size_t)s * st.nparts + b) * kMaxK + j] = cnt[0][j] + cnt[1][j] + cnt[2][j] + cnt[3][j];
}

// Scan step 1: per (column block, segment of kScanSeg parts) sum of the histograms.
static __global__ void __launch_bounds__(256) k_lbg_scan_seg(LbgState st) {
    side_chain_priority();
    const int s = blockIdx.y, g = blockIdx.x, j = threadIdx.x;
    if (st.done[s]) return;
    const int b0 = g * kScanSeg, b1 = (b0 + kScanSeg < st.nparts) ? b0 + kScanSeg : st.nparts;
    const uint32_t *h = st.hist + ((size_t)s * st.nparts + b0) * kMaxK + j;
    uint32_t sum = 0;
    uint32_t v[kScanSeg];  // all loads of the segment in flight together
#pragma unroll
    for (int u = 0; u < kScanSeg; ++u) v[u] = h[(size_t)(b0 + u < b1 ? u : b1 - 1 - b0) * kMaxK];
#pragma unroll
    for (int u = 0; u < kScanSeg; ++u) sum += (b0 + u < b1) ? v[u] : 0u;
    st.seg[((size_t)s * st.nseg + g) * kMaxK + j] = sum;
}

// Scan step 2 ("plan"): one workgroup of 256 threads per column block; thread j owns cluster j.
// Segment sums -> exclusive prefixes; per cluster: count, first position in perm, first leaf,
// rank among the empty clusters; per column block: number of leaves and of small clusters, and
// the re-seed cursor advanced by the number of empty clusters.
// Leaves: a small cluster (1..1024 members) is one leaf over its whole member list; a large
// cluster has one leaf per part, unless the streaming kernel sums the large clusters.
// Thread j of 256, in group g of as many (group 0 writes): run members of cluster j; pc, pl: its first position and leaf.
__device__ __forceinline__ void lbg_plan_clusters(const LbgState &st, int s, int j, int k, int g, uint32_t run, uint32_t &pc, uint32_t &pl) {
    __shared__ uint32_t sh_cnt[4], sh_leaf[4], sh_empty[4], sh_small[4];  // totals of the four waves
    const bool live = j < k;
    const uint32_t cnt = live ? run : 0;
    const bool small = cnt > 0 && cnt <= (uint32_t)kSeqMax;
    const bool big = cnt > (uint32_t)kSeqMax;
    const uint32_t nl = small ? 1u : ((big && !st.stream) ? (uint32_t)st.nparts : 0u);
    const uint32_t emp = (live && cnt == 0) ? 1u : 0u;
    // exclusive prefixes over j: inside a wave by shuffles, the three waves before by their totals
    // (a serial walk per thread is 4 x 255 dependent LDS reads for the last one: 10 us on this chain)
    uint32_t ic = cnt, il = nl, ie = emp, is = small ? 1u : 0u;  // inclusive inside the wave
    const int lane = j & 63, wv = j >> 6;
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
        const uint32_t oc = __shfl_up(ic, off), ol = __shfl_up(il, off), oe = __shfl_up(ie, off), os = __shfl_up(is, off);
        if (lane >= off) {
            ic += oc;
            il += ol;
            ie += oe;
            is += os;
        }
    }
    if (lane == 63) {
        sh_cnt[wv] = ic;
        sh_leaf[wv] = il;
        sh_empty[wv] = ie;
        sh_small[wv] = is;
    }
    __syncthreads();
    pc = ic - cnt;
    pl = il - nl;
    uint32_t pe = ie - emp, ps = is - (small ? 1u : 0u);
    for (int u = 0; u < wv; ++u) {
        pc += sh_cnt[u];
        pl += sh_leaf[u];
        pe += sh_empty[u];
        ps += sh_small[u];
    }
    if (g) return;
    const size_t sj = (size_t)s * kMaxK + j;
    st.count[sj] = cnt;
    st.start[sj] = pc;
    st.leaf_start[sj] = pl;
    st.empty_rank[sj] = pe;
    if (st.order) {
        st.place[sj] = small ? ps : (pl - ps) / (uint32_t)st.nparts;
        const int c = small ? long_class(cnt) : 2;  // (the counters were cleared before the barrier)
        const uint4 leaf = make_uint4(pc, pc + cnt, pl, 0u);
        if (c < 2) st.longs[((size_t)s * 2 + c) * st.long_cap + atomicAdd(&st.nlong[2 * s + c], 1)] = leaf;
        if (small) st.order[(size_t)s * st.leaf_cap + ps] = c < 2 ? make_uint4(0u, 0u, kNoLeaf, 0u) : leaf;
    } else if (small) {
        st.leaf_desc[(size_t)s * st.leaf_cap + pl] = make_uint2(pc, pc + cnt);
    }
    if (j == kMaxK - 1) {
        st.nleaves[s] = (int)(pl + nl);
        st.nsmall[s] = (int)(ps + (small ? 1u : 0u));
        int u = st.used[s];
        st.ubase[s] = u;
        st.used[s] = u + (int)(pe + emp);
        if (st.done_next) {  // the loop control of src/utils.rs:57,104-106: this update is the last one if no code changed
            st.iters[s] += 1;
            st.done_next[s] = st.changed[s] ? 0 : 1;
            st.changed[s] = 0;
        }
    }
}

static __global__ void __launch_bounds__(256) k_lbg_plan(LbgState st, int k) {
    side_chain_priority();
    const int s = blockIdx.x, j = threadIdx.x;
    if (st.done[s]) {
        if (st.done_next && j == 0) st.done_next[s] = 1;
        return;
    }
    uint32_t run = 0;
    uint32_t *h = st.seg + (size_t)s * st.nseg * kMaxK + j;
    for (int g0 = 0; g0 < st.nseg; g0 += 8) {
        uint32_t v[8];
#pragma unroll
        for (int u = 0; u < 8; ++u) v[u] = (g0 + u < st.nseg) ? h[(size_t)(g0 + u) * kMaxK] : 0u;
#pragma unroll
        for (int u = 0; u < 8; ++u) {
            if (g0 + u < st.nseg) h[(size_t)(g0 + u) * kMaxK] = run;
            run += v[u];
        }
    }
    if (st.order && j < 2) st.nlong[2 * s + j] = 0;
    uint32_t pc, pl;
    lbg_plan_clusters(st, s, j, k, 0, run, pc, pl);
}

// The three steps in one launch for up to kScanMost segments (524,288 rows) where no streaming kernel runs beside
// them: 256 threads per segment, thread j of each with its cluster's kScanSeg entries.  14 -> 6 us; beyond, a
// single workgroup cannot keep the loads of a column block in flight.
constexpr int kScanMost = 4;
static __global__ void __launch_bounds__(256 * kScanMost) k_lbg_scan(LbgState st, int k) {
    const int s = blockIdx.x, g = threadIdx.x >> 8, j = threadIdx.x & 255;
    if (st.done[s]) {
        if (st.done_next && threadIdx.x == 0) st.done_next[s] = 1;
        return;
    }
    __shared__ uint32_t sums[kScanMost][kMaxK];
    const int b0 = g * kScanSeg, b1 = (b0 + kScanSeg < st.nparts) ? b0 + kScanSeg : st.nparts;
    uint32_t *h = st.hist + ((size_t)s * st.nparts + b0) * kMaxK + j;
    uint32_t v[kScanSeg], sum = 0;
#pragma unroll
    for (int u = 0; u < kScanSeg; ++u) v[u] = h[(size_t)(b0 + u < b1 ? u : b1 - 1 - b0) * kMaxK];
#pragma unroll
    for (int u = 0; u < kScanSeg; ++u) sum += (b0 + u < b1) ? v[u] : 0u;
    sums[g][j] = sum;
    __syncthreads();
    uint32_t all = 0, run = 0;
    for (int u = 0; u < st.nseg; ++u) {
        if (u < g) run += sums[u][j];
        all += sums[u][j];
    }
    uint32_t pc, pl;
    lbg_plan_clusters(st, s, j, k, g, all, pc, pl);
    const bool leaves = j < k && !st.stream && all > (uint32_t)kSeqMax;
    uint2 *desc = st.leaf_desc + (size_t)s * st.leaf_cap + pl + (uint32_t)b0;
#pragma unroll
    for (int u = 0; u < kScanSeg; ++u) {
        if (b0 + u < b1) {
            h[(size_t)u * kMaxK] = run;
            if (leaves) desc[u] = make_uint2(pc + run, pc + run + v[u]);
            run += v[u];
        }
    }
}

// Scan step 3: per (column block, segment): histograms -> exclusive prefixes over parts (offset
// of part b inside cluster j), in place; emits the per-part leaves of the large clusters when
// they are summed by the gather path.
static __global__ void __launch_bounds__(256) k_lbg_scan_blocks(LbgState st) {
    side_chain_priority();
    const int s = blockIdx.y, g = blockIdx.x, j = threadIdx.x;
    if (st.done[s]) return;
    const int b0 = g * kScanSeg, b1 = (b0 + kScanSeg < st.nparts) ? b0 + kScanSeg : st.nparts;
    uint32_t *h = st.hist + ((size_t)s * st.nparts + b0) * kMaxK + j;
    uint32_t run = st.seg[((size_t)s * st.nseg + g) * kMaxK + j];
    const size_t sj = (size_t)s * kMaxK + j;
    const bool leaves = !st.stream && st.count[sj] > (uint32_t)kSeqMax;
    const uint32_t first = st.start[sj];
    const uint32_t leaf0 = st.leaf_start[sj] + (uint32_t)b0;  // (read here: the stores below may alias it)
    uint2 *desc = st.leaf_desc + (size_t)s * st.leaf_cap + leaf0;
    // (order: the large clusters' leaves of a part side by side)
    const int nsmall = st.order ? st.nsmall[s] : 0, nbig = st.order ? (st.nleaves[s] - nsmall) / st.nparts : 0;
    const int place = st.order ? nsmall + b0 * nbig + (int)st.place[sj] : 0;
    // the segment's entries in one memory round trip (unconditional loads, clamped to the last part)
    uint32_t v[kScanSeg];
#pragma unroll
    for (int u = 0; u < kScanSeg; ++u) v[u] = h[(size_t)(b0 + u < b1 ? u : b1 - 1 - b0) * kMaxK];
    if (st.order) {  // uniform
        uint32_t need = 0;  // this thread's long leaves of the two classes, 16 bits each; one reservation per wave and class
#pragma unroll
        for (int u = 0; u < kScanSeg; ++u) {
            const int c = leaves && b0 + u < b1 ? long_class(v[u]) : 2;
            need += c == 0 ? 1u : c == 1 ? 0x10000u : 0u;
        }
        const int lane = j & 63;
        uint32_t upto = need;  // of this lane and those before it
#pragma unroll
        for (int off = 1; off < 64; off <<= 1) {
            const uint32_t o = __shfl_up(upto, off);
            upto += lane >= off ? o : 0u;
        }
        const uint32_t all = __shfl(upto, 63);
        int base = 0;
        if (lane < 2 && all) base = atomicAdd(&st.nlong[2 * s + lane], (int)((all >> (16 * lane)) & 0xffffu));
        // the leaves at their places while the reservation is on its way
        uint4 *order = st.order + (size_t)s * st.leaf_cap + place;
        uint32_t at = first + run;
#pragma unroll
        for (int u = 0; u < kScanSeg; ++u) {
            if (b0 + u < b1 && leaves)
                order[(size_t)u * nbig] = v[u] >= kLong ? make_uint4(0u, 0u, kNoLeaf, 0u) : make_uint4(at, at + v[u], leaf0 + (uint32_t)u, 0u);
            at += v[u];
        }
        if (all) {  // uniform
            int slot0 = __shfl(base, 0) + (int)((upto - need) & 0xffffu), slot1 = __shfl(base, 1) + (int)((upto - need) >> 16);
            uint4 *longs = st.longs + (size_t)s * 2 * st.long_cap;
            at = first + run;
#pragma unroll
            for (int u = 0; u < kScanSeg; ++u) {
                if (b0 + u < b1 && leaves && v[u] >= kLong)
                    longs[v[u] >= kVeryLong ? slot0++ : st.long_cap + slot1++] = make_uint4(at, at + v[u], leaf0 + (uint32_t)u, 0u);
                at += v[u];
            }
        }
    }
#pragma unroll
    for (int u = 0; u < kScanSeg; ++u) {
        if (b0 + u < b1) {
            h[(size_t)u * kMaxK] = run;
            if (leaves && !st.order) desc[u] = make_uint2(first + run, first + run + v[u]);
            run += v[u];
        }
    }
}

// One wave per (part, column block): stable ranked scatter of row ids into perm[s].  When the
// streaming kernel sums the large clusters only the rows of small clusters are listed.
static __global__ void __launch_bounds__(64) k_lbg_scatter(LbgState st, int64_t n) {
    side_chain_priority();
    const int s = blockIdx.y, b = blockIdx.x;
    if (st.done[s]) return;
    if (st.stream && st.nsmall[s] == 0) return;
    __shared__ uint32_t base[kMaxK];
    __shared__ uint8_t listed[kMaxK];
    // codes are staged a quarter of the part at a time (16 per lane, the next quarter's load in
    // flight meanwhile): the workgroup keeps 2.3 KB of LDS and fits beside the streaming kernel
    constexpr int kStage = kPartRows / 4;
    __shared__ __attribute__((aligned(16))) uint8_t pcodes[kStage];
    const uint32_t *h = st.hist + ((size_t)s * st.nparts + b) * kMaxK;
    const uint32_t *start = st.start + (size_t)s * kMaxK;
    const uint32_t *count = st.count + (size_t)s * kMaxK;
    for (int j = threadIdx.x; j < kMaxK; j += 64) {
        base[j] = start[j] + h[j];
        listed[j] = (!st.stream || count[j] <= (uint32_t)kSeqMax) ? 1 : 0;
    }
    const uint8_t *codes = st.codes + (size_t)s * n;
    uint32_t *perm = st.perm + (size_t)s * n;
    const int lane = threadIdx.x;
    const uint64_t lt = (lane == 0) ? 0ull : (~0ull >> (64 - lane));
    int64_t lo = (int64_t)b * kPartRows;
    int64_t hi = lo + kPartRows < n ? lo + kPartRows : n;
    const bool vec = ((uintptr_t)(codes + lo) & 15) == 0;
    auto fetch = [&](int64_t q0) {  // codes of rows q0 + 16 lane .. + 15; rows from hi on read as 0, never used
        uint4 v = make_uint4(0u, 0u, 0u, 0u);
        const int64_t r0 = q0 + 16 * lane;
        if (vec && r0 + 16 <= hi) {
            v = *reinterpret_cast<const uint4 *>(codes + r0);
        } else {
            uint32_t w[4] = {0u, 0u, 0u, 0u};
            for (int u = 0; u < 16; ++u)
                if (r0 + u < hi) w[u >> 2] |= (uint32_t)codes[r0 + u] << (8 * (u & 3));
            v = make_uint4(w[0], w[1], w[2], w[3]);
        }
        return v;
    };
    uint4 ahead = fetch(lo);
    for (int64_t q0 = lo; q0 < hi; q0 += kStage) {
        __syncthreads();  // the previous quarter has been consumed (and base / listed are written)
        reinterpret_cast<uint4 *>(pcodes)[lane] = ahead;
        if (q0 + kStage < hi) ahead = fetch(q0 + kStage);
        __syncthreads();
        const int64_t qhi = q0 + kStage < hi ? q0 + kStage : hi;
        for (int64_t i0 = q0; i0 < qhi; i0 += 64) {
            int64_t i = i0 + lane;
            bool valid = i < hi;
            uint32_t c = valid ? pcodes[i - q0] : 0u;
            valid = valid && listed[c];
            uint64_t mask = __ballot(valid);
            if (mask == 0) continue;  // uniform
            if (__popcll(mask) <= 4) {
                // few listed rows (the small clusters beside the streaming kernel): one lane at a time,
                // in lane = row order; LDS operations of one wave are performed in program order
                for (uint64_t mm = mask; mm; mm &= mm - 1) {
                    if (lane == __ffsll((unsigned long long)mm) - 1) {
                        const uint32_t pos = base[c];
                        base[c] = pos + 1;
                        perm[pos] = (uint32_t)i;
                    }
                    __builtin_amdgcn_wave_barrier();
                }
                continue;
            }
    #pragma unroll
            for (int bit = 0; bit < 8; ++bit) {
                bool set = (c >> bit) & 1u;
                uint64_t bal = __ballot(set);
                mask &= set ? bal : ~bal;
            }
            // lanes with equal code and valid: mask (invalid lanes have a stale mask, unused)
            uint32_t rank = (uint32_t)__popcll(mask & lt);
            uint32_t tot = (uint32_t)__popcll(mask);
            uint32_t pos = 0;
            if (valid) pos = base[c] + rank;
            __builtin_amdgcn_wave_barrier();  // one wave, LDS in program order: reads above, updates below
            if (valid && rank == 0) base[c] += tot;
            __builtin_amdgcn_wave_barrier();
            if (valid) perm[pos] = (uint32_t)i;
        }
    }
}

// The same scatter by a workgroup of W waves per (part, column block): wave w ranks the w-th W-th of the part's
// rows.  A first sweep counts the listed codes of each share, so that a wave's first position inside
// cluster j is the part's position plus the members in the shares before its own; the order of the rows inside a
// cluster stays the row order.  A wave is a chain of 4096 / 64 W dependent LDS round trips (and there is a handful of workgroups
// on the whole GPU when there is one column block): four waves per part 13 us, sixteen 9.
constexpr int kScatterWaves = 16;

static __global__ void __launch_bounds__(64 * kScatterWaves) k_lbg_scatter_wg(LbgState st, int64_t n) {
    side_chain_priority();
    const int s = blockIdx.y, b = blockIdx.x;
    if (st.done[s]) return;
    if (st.stream && st.nsmall[s] == 0) return;
    constexpr int W = kScatterWaves, kShare = kPartRows / W;
    __shared__ uint32_t cntq[W][kMaxK];
    __shared__ uint8_t listed[kMaxK];
    __shared__ __attribute__((aligned(16))) uint8_t pcodes[kPartRows];
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const uint8_t *codes = st.codes + (size_t)s * n;
    uint32_t *perm = st.perm + (size_t)s * n;
    const int64_t lo = (int64_t)b * kPartRows;
    const int64_t hi = lo + kPartRows < n ? lo + kPartRows : n;
    const int rows = (int)(hi - lo);
    for (int j = threadIdx.x; j < W * kMaxK; j += 64 * W) (&cntq[0][0])[j] = 0u;
    if (threadIdx.x < kMaxK)
        listed[threadIdx.x] = (!st.stream || st.count[(size_t)s * kMaxK + threadIdx.x] <= (uint32_t)kSeqMax) ? 1 : 0;
    // the part's codes into LDS, 16 per thread
    if (threadIdx.x < kPartRows / 16) {
        const int64_t r0 = lo + 16 * (int64_t)threadIdx.x;
        uint4 v = make_uint4(0u, 0u, 0u, 0u);
        if (((uintptr_t)(codes + lo) & 15) == 0 && r0 + 16 <= hi) {
            v = *reinterpret_cast<const uint4 *>(codes + r0);
        } else {
            uint32_t q[4] = {0u, 0u, 0u, 0u};
            for (int u = 0; u < 16; ++u)
                if (r0 + u < hi) q[u >> 2] |= (uint32_t)codes[r0 + u] << (8 * (u & 3));
            v = make_uint4(q[0], q[1], q[2], q[3]);
        }
        reinterpret_cast<uint4 *>(pcodes)[threadIdx.x] = v;
    }
    __syncthreads();
    const int q0 = w * kShare, q1 = q0 + kShare < rows ? q0 + kShare : rows;
    for (int i = q0 + lane; i < q1; i += 64) {
        const uint32_t c = pcodes[i];
        if (listed[c]) atomicAdd(&cntq[w][c], 1u);
    }
    __syncthreads();
    if (threadIdx.x < kMaxK) {
        const uint32_t *h = st.hist + ((size_t)s * st.nparts + b) * kMaxK;
        const uint32_t *start = st.start + (size_t)s * kMaxK;
        const int j = threadIdx.x;
        uint32_t run = start[j] + h[j];
#pragma unroll
        for (int q = 0; q < W; ++q) {
            const uint32_t c = cntq[q][j];
            cntq[q][j] = run;
            run += c;
        }
    }
    __syncthreads();
    uint32_t *mybase = cntq[w];
    const uint64_t lt = (lane == 0) ? 0ull : (~0ull >> (64 - lane));
    for (int i0 = q0; i0 < q1; i0 += 64) {
        const int i = i0 + lane;
        bool valid = i < q1;
        const uint32_t c = valid ? pcodes[i] : 0u;
        valid = valid && listed[c];
        uint64_t mask = __ballot(valid);
        if (mask == 0) continue;  // uniform
#pragma unroll
        for (int bit = 0; bit < 8; ++bit) {
            const bool set = (c >> bit) & 1u;
            const uint64_t bal = __ballot(set);
            mask &= set ? bal : ~bal;
        }
        // lanes with equal code and valid: mask (invalid lanes have a stale mask, unused)
        const uint32_t rank = (uint32_t)__popcll(mask & lt);
        const uint32_t tot = (uint32_t)__popcll(mask);
        uint32_t pos = 0;
        if (valid) pos = mybase[c] + rank;
        __builtin_amdgcn_wave_barrier();  // one wave per table, LDS in program order: reads above, updates below
        if (valid && rank == 0) mybase[c] += tot;
        __builtin_amdgcn_wave_barrier();
        if (valid) perm[pos] = (uint32_t)(lo + i);
    }
}

// One lane per (leaf, component): sequential sum of the leaf's members in list order.
static __global__ void __launch_bounds__(256) k_lbg_leafsum(LbgState st, const float *__restrict__ x,
                                                     int64_t n, int64_t ld, int sd) {
    const int s = blockIdx.y;
    if (st.done[s]) return;
    int64_t gid = (int64_t)blockIdx.x * 256 + threadIdx.x;
    int64_t leaf = gid / sd;
    int t = (int)(gid % sd);
    if (leaf >= st.nleaves[s]) return;
    uint2 d = st.leaf_desc[(size_t)s * st.leaf_cap + leaf];
    const uint32_t *__restrict__ perm = st.perm + (size_t)s * n;
    const float *__restrict__ xc = x + (int64_t)s * sd + t;
    float acc = 0.0f;
    // Batches of 16 members: the loads of a batch are independent (issued unconditionally, a batch
    // past the end of the list repeats its last row and is not added), the adds stay in list order;
    // the row ids of the next batch are fetched while the current rows are in flight.
    constexpr int B = 16;
    uint32_t rn[B];
    if (d.x == d.y) {  // a large cluster has a leaf for every part, also where it has no member: nothing to read
        st.leaf_sum[((size_t)s * st.leaf_cap + leaf) * sd + t] = 0.0f;
        return;
    }
    const uint32_t lastp = d.y - 1;
#pragma unroll
    for (int u = 0; u < B; ++u) rn[u] = perm[d.x + u < d.y ? d.x + u : lastp];
    for (uint32_t p = d.x; p < d.y; p += B) {
        float v[B];
#pragma unroll
        for (int u = 0; u < B; ++u) v[u] = xc[(int64_t)rn[u] * ld];
#pragma unroll
        for (int u = 0; u < B; ++u) rn[u] = perm[p + B + u < d.y ? p + B + u : lastp];
        const uint32_t cnt = d.y - p;  // the same in every lane of the leaf
#pragma unroll
        for (int u = 0; u < B; ++u)
            if ((uint32_t)u < cnt) acc = acc + v[u];
    }
    st.leaf_sum[((size_t)s * st.leaf_cap + leaf) * sd + t] = acc;
}

// Wide column blocks: one workgroup per leaf, a lane per component, sixteen members in flight and the next sixteen
// behind them; the adds stay in list order.  What bounds it is HBM, if the rows of the leaves in flight lie together and
// no leaf is left for the end: the long leaves come first (a cluster that takes a third of the rows has 1,600 of a
// part's 4096: a chain of 100 memory round trips), then the others part by part.  Cluster by cluster, as
// k_lbg_leafsum takes them, the workgroups read all over the rows at once: 1M x 256, k = 256, with the cluster
// sizes of a residual fit's eight stages 225-240 us per pass against 185-205; in the fit 259 -> 208, which is 53.5 ->
// 50.1 ms for its eight stages with k_lbg_scan_blocks at 11 us instead of 5.5.  (Workgroups that stay and draw
// leaves from a counter: 230-550 us, the draws are in the way; the workgroups past the last leaf cost nothing.)
static __global__ void __launch_bounds__(256) k_lbg_leafsum_wide(LbgState st, const float *__restrict__ x, int64_t n,
                                                                 int64_t ld, int sd) {
    const int s = blockIdx.y;
    if (st.done[s]) return;
    const int n0 = st.nlong[2 * s], n1 = st.nlong[2 * s + 1], i = (int)blockIdx.x - n0 - n1;
    if (i >= st.nleaves[s]) return;
    const uint4 *longs = st.longs + (size_t)s * 2 * st.long_cap;
    const uint4 e = i >= 0 ? st.order[(size_t)s * st.leaf_cap + i] : longs[(int)blockIdx.x < n0 ? (int)blockIdx.x : st.long_cap + i + n1];
    const uint32_t lo = (uint32_t)__builtin_amdgcn_readfirstlane((int)e.x), hi = (uint32_t)__builtin_amdgcn_readfirstlane((int)e.y);
    if (e.z == kNoLeaf) return;
    const int t = (int)blockIdx.z * (int)blockDim.x + (int)threadIdx.x, lane = threadIdx.x & 63;
    const uint32_t *__restrict__ perm = st.perm + (size_t)s * n;
    const float *__restrict__ xc = x + (int64_t)s * sd + (t < sd ? t : 0);
    float acc = 0.0f;
    if (lo != hi) {  // (a part may have no member of a large cluster: zero, nothing to read)
        constexpr int B = 16;
        float a[B], b[B];
        const uint32_t count = hi - lo;
        uint32_t ids = 0;  // of 64 members, one per lane
        auto rows = [&](uint32_t m, float(&v)[B]) {  // past the end: the last member's again, not added
            if ((m & 63u) == 0) ids = perm[lo + m + lane < hi ? lo + m + lane : hi - 1];
#pragma unroll
            for (int u = 0; u < B; ++u) v[u] = xc[(int64_t)(uint32_t)__builtin_amdgcn_readlane((int)ids, (int)(m & 63u) + u) * ld];
        };
        rows(0, a);
        for (uint32_t m = 0; m < count; m += 2 * B) {
            if (m + B < count) rows(m + B, b);
#pragma unroll
            for (int u = 0; u < B; ++u)
                if (m + u < count) acc = acc + a[u];
            if (m + 2 * B < count) rows(m + 2 * B, a);
#pragma unroll
            for (int u = 0; u < B; ++u)
                if (m + B + u < count) acc = acc + b[u];
        }
    }
    if (t < sd) st.leaf_sum[((size_t)s * st.leaf_cap + e.z) * sd + t] = acc;
}

// A workgroup per leaf and tile of components (grid z); the last tile begins at the block's end less its width.
template <int NT, int VEC>
static __global__ void __launch_bounds__(NT) k_lbg_leafsum_tile(LbgState st, const float *__restrict__ x, int64_t n, int64_t ld,
                                                                int sd, int width, int pieces) {
    const int s = blockIdx.y;
    if (st.done[s]) return;
    const int64_t leaf = blockIdx.x;
    if (leaf >= st.nleaves[s]) return;  // uniform per workgroup
    extern __shared__ float4 lds_tile[];
    const int first = (int)blockIdx.z * width < sd - width ? (int)blockIdx.z * width : sd - width;
    const uint2 d = st.leaf_desc[(size_t)s * st.leaf_cap + leaf];
    const uint32_t *__restrict__ perm = st.perm + (size_t)s * n;
    const float acc = member_tile_sum<NT, VEC>(reinterpret_cast<float *>(lds_tile), x + (int64_t)s * sd + first, ld, d.x, d.y, width, pieces,
                                               [&](uint32_t p) { return perm[p]; });
    if ((int)threadIdx.x < width) st.leaf_sum[((size_t)s * st.leaf_cap + leaf) * sd + first + threadIdx.x] = acc;
}

// Few, long leaves (the small clusters beside the streaming kernel: up to 1024 members each): one
// workgroup per leaf.  All 256 threads fetch the members of a chunk (row ids, then 16-byte pieces
// of the sub-vectors, every load of the chunk in flight together) and store them transposed in
// LDS; lanes 0..sub_dim-1 of wave 0 then add them in list order, four members per LDS read.  The
// chain of dependent adds is the only serial part left.
constexpr int kLeafWgFloats = 8192;  // floats staged per chunk

static __global__ void __launch_bounds__(256) k_lbg_leafsum_wg(LbgState st, const float *__restrict__ x, int64_t n,
                                                               int64_t ld, int sd, int sd_shift) {
    side_chain_priority();
    const int s = blockIdx.y;
    if (st.done[s]) return;
    const int64_t leaf = blockIdx.x;
    if (leaf >= st.nleaves[s]) return;  // uniform per workgroup
    __shared__ float stage[kLeafWgFloats + 4 * 32];
    const int tid = threadIdx.x;
    const uint2 d = st.leaf_desc[(size_t)s * st.leaf_cap + leaf];
    const uint32_t *__restrict__ perm = st.perm + (size_t)s * n;
    const float *__restrict__ xs = x + (int64_t)s * sd;
    const uint32_t chunk = (uint32_t)(kLeafWgFloats >> sd_shift);  // members per chunk, a multiple of 4
    const uint32_t stride = chunk + 4;                             // floats per component row in LDS
    const int pshift = sd_shift - 2;                               // 16-byte pieces per member: 1 << pshift
    constexpr int E = kLeafWgFloats / 4 / 256;                     // pieces per thread and chunk
    float acc = 0.0f;
    for (uint32_t p = d.x; p < d.y; p += chunk) {
        const uint32_t cm = (d.y - p < chunk) ? d.y - p : chunk;
        const uint32_t tot = cm << pshift;
        uint32_t row[E];
        float4 v[E];
#pragma unroll
        for (int i = 0; i < E; ++i) {
            const uint32_t e = (uint32_t)tid + 256u * i;
            row[i] = (e < tot) ? perm[p + (e >> pshift)] : 0u;
        }
#pragma unroll
        for (int i = 0; i < E; ++i) {
            const uint32_t e = (uint32_t)tid + 256u * i;
            const uint32_t piece = e & ((1u << pshift) - 1u);
            v[i] = (e < tot) ? *reinterpret_cast<const float4 *>(xs + (int64_t)row[i] * ld + 4 * piece)
                             : make_float4(0.f, 0.f, 0.f, 0.f);
        }
        __syncthreads();  // the previous chunk has been added
#pragma unroll
        for (int i = 0; i < E; ++i) {
            const uint32_t e = (uint32_t)tid + 256u * i;
            if (e < tot) {
                const uint32_t mbr = e >> pshift, t0 = 4 * (e & ((1u << pshift) - 1u));
                stage[(t0 + 0) * stride + mbr] = v[i].x;
                stage[(t0 + 1) * stride + mbr] = v[i].y;
                stage[(t0 + 2) * stride + mbr] = v[i].z;
                stage[(t0 + 3) * stride + mbr] = v[i].w;
            }
        }
        __syncthreads();
        if (tid < sd) {
            const float *mine = stage + (size_t)tid * stride;
            uint32_t mbr = 0;
            for (; mbr + 16 <= cm; mbr += 16) {
                float4 q[4];
#pragma unroll
                for (int u = 0; u < 4; ++u) q[u] = *reinterpret_cast<const float4 *>(mine + mbr + 4 * u);
#pragma unroll
                for (int u = 0; u < 4; ++u) {
                    acc = acc + q[u].x;
                    acc = acc + q[u].y;
                    acc = acc + q[u].z;
                    acc = acc + q[u].w;
                }
            }
            for (; mbr < cm; ++mbr) acc = acc + mine[mbr];
        }
    }
    if (tid < sd) st.leaf_sum[((size_t)s * st.leaf_cap + leaf) * sd + tid] = acc;
}

// One lane per (cluster, component): the mean of a small cluster, the sequential fold over the
// per-part leaves of a large one (gather path), or the re-seed row of an empty cluster
// (src/vector.rs:315-316, src/utils.rs:98-101).
static __global__ void __launch_bounds__(256) k_lbg_finalize(LbgState st, const float *__restrict__ x,
                                                      int64_t ld, int k, int sd,
                                                      const uint32_t *__restrict__ reseed,
                                                      int n_reseed, float *__restrict__ cb) {
    const int s = blockIdx.y;
    if (st.done[s]) return;
    int64_t gid = (int64_t)blockIdx.x * 256 + threadIdx.x;
    int j = (int)(gid / sd);
    int t = (int)(gid % sd);
    if (j >= k) return;
    const size_t sj = (size_t)s * kMaxK + j;
    uint32_t cnt = st.count[sj];
    float *out = cb + ((size_t)s * k + j) * sd + t;
    if (cnt == 0) {
        int pos = st.ubase[s] + (int)st.empty_rank[sj];
        if (pos >= n_reseed) {
            st.err[0] = 1;
            return;
        }
        uint32_t r = reseed[(size_t)s * n_reseed + pos];
        *out = x[(int64_t)r * ld + (int64_t)s * sd + t];
        return;
    }
    const float *ls = st.leaf_sum + ((size_t)s * st.leaf_cap + st.leaf_start[sj]) * sd + t;
    float sum;
    if (cnt <= (uint32_t)kSeqMax) {
        sum = ls[0];
    } else {
        if (st.stream) return;  // k_lbg_combine8 writes the large clusters
        // the per-part sums in part order; 64 loads in flight (the kernel's time is memory round
        // trips; with 245 parts of a million rows the 64 MB of leaf sums then come in at the HBM rate),
        // the adds one chain
        sum = 0.0f;
        constexpr int B = 64;
        const int np = st.nparts;
        for (int p = 0; p < np; p += B) {
            float v[B];
#pragma unroll
            for (int u = 0; u < B; ++u) v[u] = ls[(size_t)(p + u < np ? p + u : np - 1) * sd];
#pragma unroll
            for (int u = 0; u < B; ++u)
                if (p + u < np) sum = sum + v[u];
        }
    }
    *out = sum / __uint2float_rn(cnt);
}

// ---- the whole update of a small fit in one launch ------------------------------------------------
// Below some ten thousand rows every kernel of the path above is a handful of waves and the update is
// a chain of launches and memory round trips: 75 us per iteration at 10,000 x 128, m = 16, k = 256 (the
// streaming kernel's 12 workgroups 47 of them), 9.8 us here; 30 us at 50,000 rows.  Here a workgroup owns C clusters of one column block:
// it reads all codes of the block, lists the rows of its own clusters in row order, sorts a window of
// the list by cluster (a stable counting sort by ballots), brings the window's sub-vectors into LDS
// (every load of up to 8192 floats in flight together), and one lane per (cluster, component) adds
// them in list order (add_members).  The orders of summation are those above: row order up
// to 1024 members, part sums in part order above.
// DEFER: clusters above 1024 members are counted and left to k_lbg_large.
// Blocks above 32 floats (TILES, of SD 16 or 32): a workgroup takes a tile of the components of C clusters.  The floats that it
// brings in are those of a whole block of C / tiles clusters, but a stage holds 1024 or 512 members instead of 170 of 96 floats, and a
// long cluster's are spread over several workgroups: what bounded it was one memory round trip per stage of the longest cluster.
// An iteration of a residual fit of 6,264 x 96, k = 186 61 -> 49 us, 7,143 x 100, k = 214 87 -> 63; fits, three or four stages of six iterations, of
// 8,000 x 256, k = 256 2330 -> 1645 us, 10,000 x 512 2709 -> 1797, 12,000 x 300, k = 100 3536 -> 2273.
// STAGED: sub_dim a multiple of 4 up to 512, a thread per component.  Else (wider blocks) a wave takes
// one cluster and 64 components at a time and reads the rows themselves, 16 rows in flight.
constexpr int kSmallList = 8192;    // listed rows held before the list is worked off: at least 16 per thread
constexpr int kSmallThreads = 512;  // one workgroup per compute unit: eight waves
constexpr int kSmallWindow = 4 * kSmallThreads;  // listed rows sorted at a time
constexpr int kSmallClusters = 16;  // most clusters per workgroup: four bits of a list entry
constexpr int kSmallWaves = kSmallThreads / 64;
constexpr int kSmallStage = 32 * kSmallThreads;  // floats staged at a time: eight 16-byte loads per thread in flight

// Workgroup number -> index such that each XCD (workgroups are dealt to the 8 XCDs in turn) gets a
// contiguous range: the workgroups that read the same codes and the same lines share an L2.
__device__ __forceinline__ unsigned xcd_contiguous(unsigned id, unsigned total) {
    const unsigned per = total / 8u, rest = total % 8u, xcd = id % 8u;
    return xcd * per + (xcd < rest ? xcd : rest) + id / 8u;
}

// The loop control of src/utils.rs:57,104-106 needs no launch of its own: every iteration has its own
// flags.  changed[it][s], it >= 1: a code of block s changed in iteration it - 1 (changed[0] is all
// ones); a block whose flag is 0 has converged, and its later flags then stay 0.  empties[it][s]: empty
// clusters re-seeded in iteration it, whose sum over the iterations before is the block's place in
// its re-seed stream.
struct LbgSmall {
    int *changed;    // [max_iters + 1][m]
    int *empties;    // [max_iters][m]
    int *err;        // 1   set to 1 when a re-seed stream runs out
    uint8_t *codes;  // [m][n]
    // wide blocks: the clusters above 1024 members, left to k_lbg_large
    int *n_large;        // [max_iters]
    uint2 *large;        // [most of an iteration]  {s * 256 + cluster, members}
    int *arrived;        // [most of an iteration]  parts summed
    float *large_sum;    // [most of an iteration][nparts][sd]
};

// codes = 0 (src/utils.rs:55), the flags, and the initial centroids x[idx[s][j]] (src/utils.rs:54; with
// pend_cb, one column block: the row as the pending residual update will leave it).
static __global__ void __launch_bounds__(256) k_lbg_small_init(LbgSmall st, const float *__restrict__ x, int64_t n,
                                                               int64_t ld, int m, int k, int sd, int max_iters, int most_large,
                                                               const uint32_t *__restrict__ idx, float *__restrict__ cb,
                                                               const float *__restrict__ pend_cb,
                                                               const uint8_t *__restrict__ pend_codes) {
    const int64_t i0 = (int64_t)blockIdx.x * 256 + threadIdx.x, stride = (int64_t)gridDim.x * 256;
    for (int64_t i = i0; i < (int64_t)m * k * sd; i += stride) {
        const int t = (int)(i % sd);
        const int64_t sj = i / sd;
        const uint32_t row = idx[sj];
        const float v = x[(int64_t)row * ld + (sj / k) * sd + t];
        cb[i] = pend_cb ? v - pend_cb[(size_t)pend_codes[row] * sd + t] : v;
    }
    for (int64_t i = i0; i < ((int64_t)m * n + 3) / 4; i += stride) reinterpret_cast<uint32_t *>(st.codes)[i] = 0u;
    // (changed, empties, err, n_large, arrived lie one behind the other)
    for (int64_t i = i0; i < (int64_t)(2 * max_iters + 1) * m + 1 + max_iters + most_large; i += stride)
        st.changed[i] = i < m ? 1 : 0;
}

// The flags to page-locked host memory.
static __global__ void __launch_bounds__(256) k_lbg_small_report(const int *__restrict__ flags, int count, int *out) {
    for (int i = threadIdx.x; i < count; i += 256) out[i] = flags[i];
}

// Which sums of a cluster's members are kept: in row order; by parts for the clusters above 1024 members;
// or both, while the sizes are not known yet.
enum { kRows, kParts, kBoth };

// The members at positions i .. hi - 1 of the stage d[position][sd], rows in `row`, onto one (cluster,
// component)'s sums: `part`, or (closed parts `total`, open part `part`) where `big`, a part closing where
// the row leaves it; kBoth: and `seq` in row order.  One chain of additions bounds a stage, that of its
// largest cluster: the next eight values are read while eight are added, at offsets that the instruction
// holds where sd is known (SD of k_lbg_update_small).  A member took 12 ns with one batch at a time,
// computed offsets and both sums in every cluster; with this, and the codes of three steps in flight instead
// of one, the first update of 60,007 rows, m = 10, k = 200, blocks of 16, whose clusters are uneven, went from
// 72.8 to 46.7 us (12.7 the list, 5 the sort, 12 the rows, 16 the sums), 60,000 rows, m = 32, blocks of 4, from
// 79.0 to 66.2, m = 4, blocks of 32, from 83.7 to 65.7.
template <int SUMS>
__device__ __forceinline__ void add_members(const float *d, int sd, const uint32_t *row, uint32_t i, uint32_t hi, bool big,
                                            float &seq, float &total, float &part, uint32_t &open) {
    constexpr int B = 8;
    auto load = [&](float (&t)[B], uint32_t &last, uint32_t at) {
        const float *b = d + at * (uint32_t)sd;
#pragma unroll
        for (int u = 0; u < B; ++u) t[u] = b[u * sd];
        if constexpr (SUMS != kRows) last = row[at + B - 1] / (uint32_t)kPartRows;
    };
    auto add_one = [&](float v, uint32_t r) {
        const uint32_t p = big ? r / (uint32_t)kPartRows : open;
        const bool close = p != open;
        const float closed = total + part;
        total = close ? closed : total;
        part = close ? 0.0f : part;
        open = p;
        part = part + v;
        if constexpr (SUMS == kBoth) seq = seq + v;
    };
    auto add = [&](const float (&t)[B], uint32_t last, uint32_t at) {
        // (rows ascend: the last one in the open part means all eight)
        if (SUMS != kRows && big && last != open) {
#pragma unroll
            for (int u = 0; u < B; ++u) add_one(t[u], row[at + u]);
        } else {
#pragma unroll
            for (int u = 0; u < B; ++u) {
                part = part + t[u];
                if constexpr (SUMS == kBoth) seq = seq + t[u];
            }
        }
    };
    float t[B], q[B];
    uint32_t last_t = 0, last_q = 0;
    if (i + B <= hi) {
        load(t, last_t, i);
        for (; i + 3 * B <= hi; i += 2 * B) {
            load(q, last_q, i + B);
            add(t, last_t, i);
            load(t, last_t, i + 2 * B);
            add(q, last_q, i + B);
        }
        if (i + 2 * B <= hi) {
            load(q, last_q, i + B);
            add(t, last_t, i);
            i += B;
            add(q, last_q, i);
        } else {
            add(t, last_t, i);
        }
        i += B;
    }
    if (i >= hi) return;
#pragma unroll
    for (int u = 0; u < B; ++u) t[u] = d[(i + u < hi ? i + u : hi - 1) * (uint32_t)sd];
#pragma unroll
    for (int u = 0; u < B; ++u) {
        if constexpr (SUMS == kRows) part = part + (i + u < hi ? t[u] : -0.0f);  // (a + -0 is a)
        else if (i + u < hi) add_one(t[u], row[i + u]);
    }
}

// The sum of v over the lanes up to this one.
__device__ __forceinline__ uint32_t wave_prefix(uint32_t v) {
    auto up = [&](auto ctrl, auto rows) {
        v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, decltype(ctrl)::value, decltype(rows)::value, 0xf, false);
    };
    up(std::integral_constant<int, 0x111>{}, std::integral_constant<int, 0xf>{});  // inside rows of 16 lanes
    up(std::integral_constant<int, 0x112>{}, std::integral_constant<int, 0xf>{});
    up(std::integral_constant<int, 0x114>{}, std::integral_constant<int, 0xf>{});
    up(std::integral_constant<int, 0x118>{}, std::integral_constant<int, 0xf>{});
    up(std::integral_constant<int, 0x142>{}, std::integral_constant<int, 0xa>{});  // lane 15 of a row to the odd row after it
    up(std::integral_constant<int, 0x143>{}, std::integral_constant<int, 0xc>{});  // lane 31 to the upper half
    return v;
}

template <bool STAGED, bool DEFER = false, int SD = 0, bool TILES = false>
static __global__ void __launch_bounds__(kSmallThreads) k_lbg_update_small(LbgSmall st, int it, int m,
                                                                           const float *__restrict__ x, int64_t n,
                                                                           int64_t ld, int sub_dim, int k, int C,
                                                                           int groups, const uint32_t *__restrict__ reseed,
                                                                           int n_reseed, float *__restrict__ cb, int tiles) {
    const int sd = SD ? SD : sub_dim, full = TILES ? sub_dim : sd;
    const unsigned id = xcd_contiguous(blockIdx.x, gridDim.x), unit = TILES ? id / (unsigned)tiles : id;  // (tiles of the same rows side by side)
    const int tile = TILES ? (int)(id % (unsigned)tiles) : 0, c0 = tile * sd < full - sd ? tile * sd : full - sd;
    const int s = (int)(unit / (unsigned)groups), j0 = (int)(unit % (unsigned)groups) * C;
    if (st.changed[it * m + s] == 0) return;  // converged before this iteration
    const int jn = k - j0 < C ? k - j0 : C;
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    __shared__ uint32_t list[kSmallList];          // row | cluster << 28
    __shared__ uint32_t sorted[kSmallWindow];      // the window's rows, cluster by cluster
    __shared__ uint32_t hist[kSmallWindow / 64][kSmallClusters];
    __shared__ uint32_t cl_off[kSmallClusters + 1];  // first position of a cluster in the sorted window
    __shared__ uint32_t cl_cnt[kSmallClusters];      // members
    __shared__ uint32_t cl_part[kSmallClusters];     // (not STAGED) part of the last member added
    __shared__ uint32_t wave_tot[2][kSmallWaves];
    extern __shared__ float dyn[];  // STAGED: the sub-vectors; else three sums per (cluster, component)
    const uint8_t *codes = st.codes + (size_t)s * n;
    const float *xs = x + (int64_t)s * full + c0;
    const uint64_t lt = lane == 0 ? 0ull : (~0ull >> (64 - lane));
    if (tid < kSmallClusters) {
        cl_cnt[tid] = 0u;
        cl_part[tid] = 0u;
    }
    if constexpr (!STAGED)
        for (int i = tid; i < 3 * C * sd; i += kSmallThreads) dyn[i] = 0.0f;
    float *sseq = dyn, *stot = dyn + C * sd, *spart = dyn + 2 * C * sd;
    // STAGED: the sums of this thread's (cluster, component): in row order; and by parts
    float seq = 0.0f, total = 0.0f, part = 0.0f;
    uint32_t cur_part = 0;
    const int my_c = STAGED ? tid / sd : 0, my_t = STAGED ? tid % sd : 0;
    const bool summing = STAGED && my_c < jn;
    int track = kRows;  // uniform
    bool drained = false;  // uniform
    bool big = false;  // STAGED: this thread's cluster is above 1024 members
    uint32_t cnt = 0;                     // entries of list, uniform

    // one member's value into (row-order sum; closed parts, open part)
    auto add_tracked = [](float v, uint32_t row, float &a, float &tt, float &pp, uint32_t &open) {
        const uint32_t p = row / (uint32_t)kPartRows;
        const bool close = p != open;
        const float closed = tt + pp;
        tt = close ? closed : tt;
        pp = close ? 0.0f : pp;
        open = p;
        a = a + v;
        pp = pp + v;
    };
    auto drain = [&]() {
        for (uint32_t w0 = 0; w0 < cnt; w0 += kSmallWindow) {
            const uint32_t wn = cnt - w0 < (uint32_t)kSmallWindow ? cnt - w0 : (uint32_t)kSmallWindow;
            // ranks inside chunks of 64 entries, chunk kSmallWaves * u + wave by this wave
            uint32_t ent[4], rank[4];
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                const uint32_t i = 64u * (kSmallWaves * u + wave) + lane;
                const bool valid = i < wn;
                ent[u] = valid ? list[w0 + i] : 0u;
                const uint32_t c = ent[u] >> 28;
                uint64_t same = __ballot(valid);
#pragma unroll
                for (int bit = 0; bit < 4; ++bit) {
                    const bool set = (c >> bit) & 1u;
                    const uint64_t bal = __ballot(set);
                    same &= set ? bal : ~bal;
                }
                rank[u] = (uint32_t)__popcll(same & lt);
                if (lane < kSmallClusters) hist[kSmallWaves * u + wave][lane] = 0u;
                __builtin_amdgcn_wave_barrier();  // one wave's LDS operations are performed in order
                if (valid && rank[u] == 0) hist[kSmallWaves * u + wave][c] = (uint32_t)__popcll(same);
            }
            __syncthreads();
            if (tid < kSmallClusters) {  // exclusive prefixes over the chunks, then over the clusters
                uint32_t h[kSmallWindow / 64], run = 0;
#pragma unroll
                for (int q = 0; q < kSmallWindow / 64; ++q) h[q] = hist[q][tid];
#pragma unroll
                for (int q = 0; q < kSmallWindow / 64; ++q) {
                    hist[q][tid] = run;
                    run += h[q];
                }
                uint32_t inc = run;
#pragma unroll
                for (int off = 1; off < kSmallClusters; off <<= 1) {
                    const uint32_t o = __shfl_up(inc, off);
                    if (tid >= off) inc += o;
                }
                cl_off[tid + 1] = inc;
                if (tid == 0) cl_off[0] = 0u;
            }
            __syncthreads();
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                const uint32_t i = 64u * (kSmallWaves * u + wave) + lane, c = ent[u] >> 28;
                if (i < wn) sorted[cl_off[c] + hist[kSmallWaves * u + wave][c] + rank[u]] = ent[u] & 0x0fffffffu;
            }
            __syncthreads();
            if constexpr (STAGED) {
                const uint32_t per = (uint32_t)sd / 4u, most = (uint32_t)kSmallStage / (uint32_t)sd;
                typedef float piece4 __attribute__((ext_vector_type(4), aligned(4)));
                constexpr int E = kSmallStage / 4 / kSmallThreads;
                piece4 v[E];
                auto gather = [&](uint32_t p0) {  // past the window's end: its first row again, not stored
                    const uint32_t pn = wn - p0 < most ? wn - p0 : most;
#pragma unroll
                    for (int e = 0; e < E; ++e) {
                        const uint32_t i = (uint32_t)tid + (uint32_t)kSmallThreads * e, ic = i < pn * per ? i : 0u;
                        v[e] = *reinterpret_cast<const piece4 *>(xs + (int64_t)sorted[p0 + ic / per] * ld + 4u * (ic % per));
                    }
                };
                gather(0);
                for (uint32_t p0 = 0; p0 < wn; p0 += most) {
                    const uint32_t pn = wn - p0 < most ? wn - p0 : most;
#pragma unroll
                    for (int e = 0; e < E; ++e) {
                        const uint32_t i = (uint32_t)tid + (uint32_t)kSmallThreads * e;
                        if (i < pn * per)
                            *reinterpret_cast<float4 *>(dyn + 4u * i) = make_float4(v[e][0], v[e][1], v[e][2], v[e][3]);
                    }
                    __syncthreads();
                    if (p0 + most < wn) gather(p0 + most);  // in flight while this stage is added
                    if (summing) {
                        const uint32_t c_lo = cl_off[my_c], c_hi = cl_off[my_c + 1];
                        uint32_t i = c_lo > p0 ? c_lo - p0 : 0u;
                        const uint32_t end = c_hi > p0 ? c_hi - p0 : 0u, hi = end < pn ? end : pn;
                        const float *d = dyn + my_t;
                        if (track == kBoth) add_members<kBoth>(d, sd, sorted + p0, i, hi, true, seq, total, part, cur_part);
                        else if (track == kParts) add_members<kParts>(d, sd, sorted + p0, i, hi, big, seq, total, part, cur_part);
                        else add_members<kRows>(d, sd, sorted + p0, i, hi, false, seq, total, part, cur_part);
                    }
                    __syncthreads();
                }
            } else {
                const int slices = (sd + 63) / 64;
                for (int task = wave; task < jn * slices; task += kSmallWaves) {
                    const int c = task / slices, t = (task % slices) * 64 + lane, tc = t < sd ? t : sd - 1;
                    const float *col = xs + tc;
                    const uint32_t lo = cl_off[c], hi = cl_off[c + 1];
                    if (lo >= hi) continue;
                    float a = sseq[c * sd + tc], tt = stot[c * sd + tc], pp = spart[c * sd + tc];
                    uint32_t open = cl_part[c];
                    constexpr int B = 16;
                    for (uint32_t i = lo; i < hi; i += B) {
                        float v[B];
                        uint32_t r[B];
#pragma unroll
                        for (int u = 0; u < B; ++u) r[u] = sorted[i + u < hi ? i + u : hi - 1];
#pragma unroll
                        for (int u = 0; u < B; ++u) v[u] = col[(int64_t)r[u] * ld];
#pragma unroll
                        for (int u = 0; u < B; ++u)
                            if (i + u < hi) {
                                if (track != kRows) add_tracked(v[u], r[u], a, tt, pp, open);
                                else a = a + v[u];
                            }
                    }
                    if (t < sd) {
                        sseq[c * sd + t] = a;
                        stot[c * sd + t] = tt;
                        spart[c * sd + t] = pp;
                    }
                }
                __syncthreads();
                if (tid < jn && cl_off[tid] < cl_off[tid + 1])
                    cl_part[tid] = sorted[cl_off[tid + 1] - 1] / (uint32_t)kPartRows;
                __syncthreads();
            }
        }
        cnt = 0;
        drained = true;
    };

    // 16 consecutive codes per thread and step, the next step's in flight
    typedef uint32_t codes16 __attribute__((ext_vector_type(4), aligned(1)));
    auto fetch = [&](int64_t r0, uint32_t &have) {
        codes16 v = {0u, 0u, 0u, 0u};
        have = r0 >= n ? 0u : (n - r0 < 16 ? (1u << (uint32_t)(n - r0)) - 1u : 0xffffu);
        if (have == 0xffffu) {
            v = *reinterpret_cast<const codes16 *>(codes + r0);
        } else if (have) {
            for (int u = 0; u < (int)(n - r0); ++u) v[u >> 2] |= (uint32_t)codes[r0 + u] << (8 * (u & 3));
        }
        return v;
    };
    constexpr int kStep = 16 * kSmallThreads;  // rows
    const int nsteps = (int)((n + kStep - 1) / kStep);
    // bit u: row row0 + u belongs to one of the workgroup's clusters
    auto own_rows = [&](const codes16 &v) {
        uint32_t mine = 0;
#pragma unroll
        for (int u = 0; u < 16; ++u) {
            const uint32_t c = (v[u >> 2] >> (8 * (u & 3))) & 0xffu;
            mine |= (c - (uint32_t)j0 < (uint32_t)jn ? 1u : 0u) << u;
        }
        return mine;
    };
    auto cluster_of = [&](const codes16 &v, uint32_t u) {
        const uint32_t w = u < 8u ? (u < 4u ? v[0] : v[1]) : (u < 12u ? v[2] : v[3]);
        return ((w >> (8u * (u & 3u))) & 0xffu) - (uint32_t)j0;
    };
    uint32_t have_next, have_2, have_3;
    codes16 next = fetch(16 * tid, have_next), next2 = fetch(kStep + 16 * tid, have_2), next3 = fetch(2 * kStep + 16 * tid, have_3);
    // the step that is next now; the one three steps on (from step p) into flight
    auto advance = [&](int64_t p) {
        next = next2;
        have_next = have_2;
        next2 = next3;
        have_2 = have_3;
        next3 = fetch((p + 3) * kStep + 16 * tid, have_3);
    };
    uint32_t large = 0;  // (DEFER) bit c: cluster j0 + c is not summed here, uniform
    if constexpr (DEFER) {
        __syncthreads();
        for (int p = 0; p < nsteps; ++p) {
            const codes16 v = next;
            uint32_t mine = own_rows(v) & have_next;
            advance(p);
            for (; mine; mine &= mine - 1) atomicAdd(&cl_cnt[cluster_of(v, (uint32_t)__ffs(mine) - 1u)], 1u);
        }
        __syncthreads();
        for (int p = -3; p < 0; ++p) advance(p);  // the first steps again
        for (int c = 0; c < jn; ++c) large |= (cl_cnt[c] > (uint32_t)kSeqMax ? 1u : 0u) << c;
        large = __builtin_amdgcn_readfirstlane(large);
        if (tile == 0 && tid < jn && ((large >> tid) & 1u))
            st.large[atomicAdd(st.n_large + it, 1)] = make_uint2((uint32_t)(s * kMaxK + j0 + tid), cl_cnt[tid]);
    }
    for (int p = 0; p < nsteps; ++p) {
        const uint32_t row0 = (uint32_t)p * (uint32_t)kStep + 16u * tid;
        const codes16 v = next;
        const uint32_t have = have_next;
        advance(p);
        uint32_t mine = own_rows(v) & have;
        if (DEFER && large)
            for (uint32_t mm = mine; mm; mm &= mm - 1)
                if ((large >> cluster_of(v, (uint32_t)__ffs(mm) - 1u)) & 1u) mine &= ~(mm & (0u - mm));
        const uint32_t m1 = __popc(mine);
        const uint32_t inc = wave_prefix(m1);
        if (lane == 63) wave_tot[p & 1][wave] = inc;
        __syncthreads();
        uint32_t before = 0, all = 0;
#pragma unroll
        for (int w = 0; w < kSmallWaves; ++w) {
            const uint32_t t = wave_tot[p & 1][w];
            before += w < wave ? t : 0u;
            all += t;
        }
        if (cnt + all > (uint32_t)kSmallList) {  // the sizes of the clusters are not known yet: keep both sums
            track = DEFER ? kRows : kBoth;
            drain();
        }
        uint32_t at = cnt + before + inc - m1;
        for (uint32_t mm = mine; mm; mm &= mm - 1) {
            const uint32_t u = (uint32_t)__ffs(mm) - 1u;
            const uint32_t c = cluster_of(v, u);
            list[at++] = (row0 + u) | (c << 28);
            if constexpr (!DEFER) atomicAdd(&cl_cnt[c], 1u);
        }
        cnt += all;
    }
    __syncthreads();
    if (!DEFER && !drained) {
        for (int c = 0; c < jn; ++c) track = cl_cnt[c] > (uint32_t)kSeqMax ? (STAGED ? kParts : kBoth) : track;
        big = summing && cl_cnt[my_c] > (uint32_t)kSeqMax;
    }
    drain();
    float *out = cb + ((size_t)s * k + j0) * full + c0;
    if constexpr (STAGED) {
        if (summing) {
            const uint32_t cm = cl_cnt[my_c];
            if (cm && !((large >> my_c) & 1u))
                out[my_c * full + my_t] =
                    (cm > (uint32_t)kSeqMax ? total + part : (track == kBoth ? seq : part)) / __uint2float_rn(cm);
        }
    } else {
        for (int i = tid; i < jn * sd; i += kSmallThreads) {
            const uint32_t cm = cl_cnt[i / sd];
            if (cm) out[i] = (cm <= (uint32_t)kSeqMax ? sseq[i] : stot[i] + spart[i]) / __uint2float_rn(cm);
        }
    }
    // Empty clusters take the next rows of the block's re-seed stream in cluster order
    // (src/utils.rs:98-101): the workgroup goes over the codes once more for the clusters that have
    // members (`list` is free by now).
    bool open = false;
    for (int c = 0; c < jn; ++c) open = open || cl_cnt[c] == 0u;
    if (!open) return;
    for (int j = tid; j < kMaxK; j += kSmallThreads) list[j] = 0u;
    __syncthreads();
    for (int64_t i = tid; i < n; i += kSmallThreads) list[codes[i]] = 1u;
    __syncthreads();
    if (tid == 0) {
        int used = 0, mine = 0;
        for (int i = 0; i < it; ++i) used += st.empties[i * m + s];
        for (int j = 0; j < j0; ++j) used += list[j] == 0u;
        for (int c = 0; c < jn; ++c) {
            cl_off[c] = (uint32_t)(used + mine);  // place in the stream
            mine += cl_cnt[c] == 0u;
        }
        if (tile == 0) atomicAdd(st.empties + it * m + s, mine);
    }
    __syncthreads();
    for (int i = tid; i < jn * sd; i += kSmallThreads) {
        const int c = i / sd, t = i % sd;
        if (cl_cnt[c]) continue;
        const int pos = (int)cl_off[c];
        if (pos >= n_reseed)
            st.err[0] = 1;  // the centroid stays
        else
            out[c * full + t] = xs[(int64_t)reseed[(size_t)s * n_reseed + pos] * ld + t];
    }
}

// The clusters above 1024 members of a small fit over wide blocks (rows that are residuals gather in a
// few of them): workgroup (part p, y) takes the listed clusters y, y + whole, ... and adds the
// members in part p in row order, staged through LDS as above; the workgroup that brings a cluster's
// last part adds the part sums in part order and divides.  One workgroup that adds such a cluster alone
// is bound by what it has in flight, 64 KB per memory round trip: 6,000 rows of 128 took 200 us.
// SD: a cluster with more than kLargeTiled members per part (three of a column block at most) is taken by tiles of SD components, which
// hold 1024 or 512 members per memory round trip: workgroups (p, whole + tile + tiles t), which look for such clusters and take the t-th, the
// (t + kLargeTurns)-th ... of them (one turn: three clusters of a block one after the other, 23,405 x 224, k = 160 95 us a launch, of 12,288 x
// 128, k = 64 55; without tiles 50 and 39).  For the others a
// fence per tile is more than what the tiles save (20,000 x 128, k = 256, tiles of all clusters 22.7 us a launch, of these 17.1;
// 15,980 x 96, k = 63 28.6 without tiles).
constexpr int kLargeTiled = 1024, kLargeTurns = 3;
template <int SD>
static __global__ void __launch_bounds__(kSmallThreads) k_lbg_large(LbgSmall st, int it, const float *__restrict__ x,
                                                                    int64_t n, int64_t ld, int full, int k, int whole,
                                                                    float *__restrict__ cb) {
    const int count = st.n_large[it];
    const bool tiled = SD != 0 && (int)blockIdx.y >= whole;
    if (tiled ? count == 0 : (int)blockIdx.y >= count) return;
    const int tiles = SD ? (full + SD - 1) / (SD ? SD : 1) : 1, tile = tiled ? ((int)blockIdx.y - whole) % tiles : 0;
    const int p = blockIdx.x, nparts = gridDim.x, tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    __shared__ uint16_t list[kPartRows];
    __shared__ uint32_t wave_tot[kSmallWaves];
    __shared__ int last;
    extern __shared__ float dyn[];
    const int64_t lo = (int64_t)p * kPartRows;
    const int rows = n - lo < kPartRows ? (int)(n - lo) : kPartRows;
    typedef float piece4 __attribute__((ext_vector_type(4), aligned(4)));
    auto by_tiles = [&](uint32_t members) { return SD != 0 && members > (uint32_t)(kLargeTiled * nparts); };
    auto cluster = [&](int e) {
        const uint2 ent = st.large[e];
        const int s = (int)(ent.x / kMaxK), c0 = !tiled ? 0 : tile * SD < full - SD ? tile * SD : full - SD;
        const uint32_t j = ent.x % kMaxK;
        const uint8_t *codes = st.codes + (size_t)s * n + lo;
        uint32_t mine = 0;  // of the thread's eight consecutive rows
#pragma unroll
        for (int u = 0; u < 8; ++u) {
            const int i = 8 * tid + u;
            mine |= (i < rows && codes[i < rows ? i : 0] == j ? 1u : 0u) << u;
        }
        uint32_t inc = __popc(mine);
        const uint32_t own = inc;
#pragma unroll
        for (int off = 1; off < 64; off <<= 1) {
            const uint32_t o = __shfl_up(inc, off);
            if (lane >= off) inc += o;
        }
        if (lane == 63) wave_tot[wave] = inc;
        __syncthreads();
        uint32_t at = inc - own, cnt = 0;
#pragma unroll
        for (int w = 0; w < kSmallWaves; ++w) {
            at += w < wave ? wave_tot[w] : 0u;
            cnt += wave_tot[w];
        }
        for (; mine; mine &= mine - 1) list[at++] = (uint16_t)(8 * tid + __ffs(mine) - 1);
        __syncthreads();
        const float *xs = x + lo * ld + (int64_t)s * full + c0;
        float sum = 0.0f;
        auto add_part = [&](auto fixed) {
            constexpr int W = decltype(fixed)::value;
            const uint32_t sd = W ? W : full, per = sd / 4u, most = (uint32_t)kSmallStage / sd;
            constexpr int E = kSmallStage / 4 / kSmallThreads;
            piece4 v[E];
            float unused = 0.0f;
            uint32_t open = 0;
            auto gather = [&](uint32_t p0) {
                const uint32_t pn = cnt - p0 < most ? cnt - p0 : most;
#pragma unroll
                for (int u = 0; u < E; ++u) {
                    const uint32_t i = (uint32_t)tid + (uint32_t)kSmallThreads * u, ic = i < pn * per ? i : 0u;
                    v[u] = *reinterpret_cast<const piece4 *>(xs + (int64_t)list[p0 + ic / per] * ld + 4u * (ic % per));
                }
            };
            if (cnt) gather(0);
            for (uint32_t p0 = 0; p0 < cnt; p0 += most) {
                const uint32_t pn = cnt - p0 < most ? cnt - p0 : most;
#pragma unroll
                for (int u = 0; u < E; ++u) {
                    const uint32_t i = (uint32_t)tid + (uint32_t)kSmallThreads * u;
                    if (i < pn * per) *reinterpret_cast<float4 *>(dyn + 4u * i) = make_float4(v[u][0], v[u][1], v[u][2], v[u][3]);
                }
                __syncthreads();
                if (p0 + most < cnt) gather(p0 + most);
                if ((uint32_t)tid < sd) add_members<kRows>(dyn + tid, (int)sd, nullptr, 0, pn, false, unused, unused, sum, open);
                __syncthreads();
            }
        };
        const int sd = tiled ? SD : full;
        if (tiled) add_part(std::integral_constant<int, SD>{});
        else add_part(std::integral_constant<int, 0>{});
        float *sums = st.large_sum + (size_t)e * nparts * full + c0;
        int *arrived = st.arrived + (size_t)e * tiles + tile;
        if (tid < sd) sums[(size_t)p * full + tid] = sum;
        __threadfence();
        __syncthreads();
        if (tid == 0) last = atomicAdd(arrived, 1) == nparts - 1;
        __syncthreads();
        if (last) {
            __threadfence();
            if (tid < sd) {
                float total = 0.0f;
                for (int q = 0; q < nparts; ++q)
                    total = total + __hip_atomic_load(sums + (size_t)q * full + tid, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                cb[((size_t)s * k + j) * full + c0 + tid] = total / __uint2float_rn(ent.y);
            }
            if (tid == 0) *arrived = 0;  // for the next iteration
        }
        __syncthreads();
    };
    if (!tiled) {
        for (int e = blockIdx.y; e < count; e += whole)
            if (!by_tiles(st.large[e].y)) cluster(e);  // uniform
        return;
    }
    int turn = ((int)blockIdx.y - whole) / tiles;
    for (int e0 = 0; e0 < count; e0 += 64) {  // every wave finds the same entries
        const bool mine = e0 + lane < count && by_tiles(st.large[e0 + lane < count ? e0 + lane : 0].y);
        for (uint64_t mask = __ballot(mine); mask; mask &= mask - 1) {
            if (turn == 0) cluster(e0 + __ffsll((unsigned long long)mask) - 1);
            turn = turn == 0 ? kLargeTurns - 1 : turn - 1;
        }
    }
}

// ---- streaming sums of the large clusters (sub_dim 8, 4 column blocks per 128 bytes) -----------
// One workgroup per (part, group of 4 column blocks); wave w of the group owns column block
// 4g + w, so the four waves together consume whole 128-byte lines of the rows.  A wave walks
// its part 64 rows at a time; a lane holds the 32-byte sub-vector of its row.  The rows of a
// chunk are ranked inside their cluster with wave ballots and added to the cluster's
// accumulator in LDS in rank order (round r: the lanes of rank r, all on different clusters) —
// so every cluster receives its rows of this part in row order, one at a time, starting from
// 0.0.  Emits the per-part sums (k_lbg_hist counts the members, on another stream at the same
// time); no floating-point atomics.  The four waves meet at a workgroup barrier before every
// chunk (the barrier waits for nothing else: the prefetches stay in flight): each of them reads
// a different 32-byte quarter of the same lines, and waves that drift apart by the length of
// their prefetch queues find those lines gone from the compute unit's cache.
// (m not a multiple of 4: the waves of the last group without a column block only keep the barriers.)
static __global__ void __launch_bounds__(256) k_lbg_stream8(LbgState st, const float *__restrict__ x, int64_t n,
                                                            int64_t ld, int m) {
    const int g = blockIdx.y, b = blockIdx.x;
    const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int s = 4 * g + w;
    __shared__ float4 acc_lo[4][kMaxK], acc_hi[4][kMaxK];  // components 0-3 and 4-7 of every cluster
    bool work = false;
    for (int u = 0; u < 4; ++u) work = work || (4 * g + u < m && !st.done[4 * g + u]);
    if (!work) return;
    float4 *alo = acc_lo[w], *ahi = acc_hi[w];
    for (int i = lane; i < kMaxK; i += 64) {
        alo[i] = make_float4(0.f, 0.f, 0.f, 0.f);
        ahi[i] = make_float4(0.f, 0.f, 0.f, 0.f);
    }
    __builtin_amdgcn_wave_barrier();
    const int64_t lo = (int64_t)b * kPartRows;
    const int64_t hi = lo + kPartRows < n ? lo + kPartRows : n;
    constexpr int PF = 3;
    const int rows = (int)(hi - lo);
    const int nchunks = (rows + 63) / 64, rows_last = rows - 64 * (nchunks - 1);
    const int nsteps = (nchunks + PF - 1) / PF * PF;  // chunk steps of the loop below, one barrier each
    if (s >= m || st.done[s]) {  // this wave's column block has stopped: it only keeps the others' barriers company
        for (int c = 0; c < nsteps; ++c) __builtin_amdgcn_s_barrier();
        return;
    }
    // The sub-vectors and codes of the next PF chunks are kept in flight: one chunk's arithmetic
    // is far shorter than a memory round trip.  The loads are unconditional and in chunk order (a
    // load under a branch, or out of order, makes the compiler wait for every load in flight at
    // the first use): a lane without a row in the part's last chunk reads that chunk's first row,
    // the fetches past the last chunk read that chunk again, and both are dropped.
    float4 b0[PF], b1[PF];
    uint8_t bc[PF];  // (bytes until they are used: widened where they are loaded, they would be waited for there)
    // Lanes 2p and 2p+1 fetch the two 16-byte halves of row p of the chunk (b0) and of row 32 + p
    // (b1): one load instruction touches each 64-byte piece of a line once instead of twice.  The
    // neighbours then swap a half, so that lane 2p owns row p and lane 2p + 1 owns row 32 + p.
    const int pr = lane >> 1, hf = lane & 1;
    const int ridx = hf ? 32 + pr : pr;  // this lane's row of a chunk
    // addresses: a scalar base per chunk plus 32-bit lane offsets (a part spans 4096 rows: the
    // host keeps the leading dimension below 2^20 floats)
    const char *xbase = reinterpret_cast<const char *>(x + lo * ld + (int64_t)s * 8);
    const uint8_t *cbase = st.codes + (size_t)s * n + lo;
    const uint32_t hoff = 16u * (uint32_t)hf;
    const uint32_t f0 = 4u * (uint32_t)pr * (uint32_t)ld + hoff, f1 = f0 + 128u * (uint32_t)ld;
    const uint32_t l0 = pr < rows_last ? f0 : hoff, l1 = 32 + pr < rows_last ? f1 : hoff;
    const uint32_t lc = ridx < rows_last ? (uint32_t)ridx : 0u;
    const int64_t chunkb = 256 * ld;  // bytes of 64 rows
    auto fetch = [&](int chunk, float4 &d0, float4 &d1, uint8_t &dc) {
        const int cc = chunk < nchunks ? chunk : nchunks - 1;  // uniform
        const bool last = cc == nchunks - 1;
        const char *xb = xbase + cc * chunkb;
        const uint8_t *cb = cbase + 64 * cc;
        d0 = *reinterpret_cast<const float4 *>(xb + (uint64_t)(last ? l0 : f0));
        d1 = *reinterpret_cast<const float4 *>(xb + (uint64_t)(last ? l1 : f1));
        dc = cb[last ? lc : (uint32_t)ridx];
    };
#pragma unroll
    for (int u = 0; u < PF; ++u) {
        fetch(u, b0[u], b1[u], bc[u]);
        __builtin_amdgcn_sched_barrier(0);
    }
    // lanes whose row comes before this lane's row
    const unsigned long long even = 0x5555555555555555ull, below = (lane == 0) ? 0ull : (~0ull >> (64 - lane));
    const unsigned long long ltm = hf ? (even | (~even & below)) : (even & below);
    const uint32_t lt_lo = (uint32_t)ltm, lt_hi = (uint32_t)(ltm >> 32);
    for (int base = 0; base < nsteps; base += PF) {
#pragma unroll
        for (int u = 0; u < PF; ++u) {
            // (a chunk past the part's end has no pending lane and falls through: an exit from here,
            // which the compiler routes past the loop's head, would make it wait there for every
            // load in flight)
            __builtin_amdgcn_s_barrier();  // step base + u of nsteps
            const bool pending = 64 * (base + u) + ridx < rows;
            const float4 fa = b0[u], fb = b1[u];
            uint32_t c = pending ? (uint32_t)bc[u] : 0u;
            // swap: the even lane sends its half of row 32 + p, the odd lane its half of row p
            const float4 snd = hf ? fa : fb;
            float4 rcv;
            rcv.x = __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(snd.x), 0xB1, 0xF, 0xF, true));
            rcv.y = __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(snd.y), 0xB1, 0xF, 0xF, true));
            rcv.z = __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(snd.z), 0xB1, 0xF, 0xF, true));
            rcv.w = __int_as_float(__builtin_amdgcn_mov_dpp(__float_as_int(snd.w), 0xB1, 0xF, 0xF, true));
            float4 v0 = hf ? rcv : fa;  // components 0-3 of this lane's row
            float4 v1 = hf ? fb : rcv;  // components 4-7
            // the slot's registers are free from here on (the empty statement pins the selects
            // above it): its next loads go out now
            asm volatile("" : "+v"(v0.x), "+v"(v0.y), "+v"(v0.z), "+v"(v0.w), "+v"(v1.x), "+v"(v1.y), "+v"(v1.z),
                         "+v"(v1.w), "+v"(c));
            fetch(base + u + PF, b0[u], b1[u], bc[u]);
            __builtin_amdgcn_sched_barrier(0);
            // Lanes of the same cluster, found with one wave ballot per code bit: a lane differs
            // from lane j when some bit of its code differs from j's bit in the ballot.
            const unsigned long long vb = __ballot(pending);
            uint32_t bad_lo = ~(uint32_t)vb, bad_hi = ~(uint32_t)(vb >> 32);
#pragma unroll
            for (int bit = 0; bit < 8; bit += 2) {
                const int sp0 = (int)(c << (31 - bit)) >> 31, sp1 = (int)(c << (30 - bit)) >> 31;  // 0 or -1
                const unsigned long long bal0 = __ballot(sp0 != 0), bal1 = __ballot(sp1 != 0);
                bad_lo = bad_lo | ((uint32_t)bal0 ^ (uint32_t)sp0) | ((uint32_t)bal1 ^ (uint32_t)sp1);
                bad_hi = bad_hi | ((uint32_t)(bal0 >> 32) ^ (uint32_t)sp0) | ((uint32_t)(bal1 >> 32) ^ (uint32_t)sp1);
            }
            const uint32_t same_lo = ~bad_lo, same_hi = ~bad_hi;
            const uint32_t rank =
                pending ? (uint32_t)(__popc(same_lo & lt_lo) + __popc(same_hi & lt_hi)) : 0xFFFFFFFFu;
            // Round r: the lanes of rank r (all on different clusters) add their rows.  LDS
            // operations of one wave are performed in program order, so the next round sees these
            // writes; the wave barrier only pins the compiler's schedule (a fence or s_barrier
            // here would also wait for the row prefetches in flight).
            for (uint32_t r = 0; __any(rank != 0xFFFFFFFFu && rank >= r); ++r) {
                if (rank == r) {
                    float4 a0 = alo[c], a1 = ahi[c];
                    a0.x = a0.x + v0.x;
                    a0.y = a0.y + v0.y;
                    a0.z = a0.z + v0.z;
                    a0.w = a0.w + v0.w;
                    a1.x = a1.x + v1.x;
                    a1.y = a1.y + v1.y;
                    a1.z = a1.z + v1.z;
                    a1.w = a1.w + v1.w;
                    alo[c] = a0;
                    ahi[c] = a1;
                }
                __builtin_amdgcn_wave_barrier();
            }
        }
    }
    __builtin_amdgcn_wave_barrier();
    float4 *ps = reinterpret_cast<float4 *>(st.part_sum) + ((size_t)s * st.nparts + b) * kMaxK * 2;
    for (int i = lane; i < kMaxK * 2; i += 64) ps[i] = (i & 1) ? ahi[i >> 1] : alo[i >> 1];
}

// One lane per (cluster, component): sequential fold of the per-part sums of a large cluster.
static __global__ void __launch_bounds__(256) k_lbg_combine8(LbgState st, int k, float *__restrict__ cb) {
    const int s = blockIdx.y;
    if (st.done[s]) return;
    const int gid = blockIdx.x * 256 + threadIdx.x;
    const int j = gid / 8, t = gid % 8;
    if (j >= k) return;
    const uint32_t cnt = st.count[(size_t)s * kMaxK + j];
    if (cnt <= (uint32_t)kSeqMax) return;
    const float *ps = st.part_sum + ((size_t)s * st.nparts * kMaxK + j) * 8 + t;
    // the kernel is a handful of waves: its time is memory round trips, so 32 loads are in flight
    // at a time (unconditional, clamped to the last part); the adds stay one chain in part order
    float sum = 0.0f;
    constexpr int B = 32;
    const int np = st.nparts;
    for (int p = 0; p < np; p += B) {
        float v[B];
#pragma unroll
        for (int u = 0; u < B; ++u) v[u] = ps[(size_t)(p + u < np ? p + u : np - 1) * kMaxK * 8];
#pragma unroll
        for (int u = 0; u < B; ++u)
            if (p + u < np) sum = sum + v[u];
    }
    cb[((size_t)s * k + j) * 8 + t] = sum / __uint2float_rn(cnt);
}

// The same fold for every cluster, sum only (big_sum[s][j][t]): it needs nothing from the gather
// path, so it can follow the streaming kernel at once; k_lbg_finalize_prep8 picks the large
// clusters' sums and divides.
static __global__ void __launch_bounds__(256) k_lbg_fold8(LbgState st, int k, float *__restrict__ big_sum) {
    const int s = blockIdx.y;
    if (st.done[s]) return;
    const int gid = blockIdx.x * 256 + threadIdx.x;
    const int j = gid / 8, t = gid % 8;
    if (j >= k) return;
    const float *ps = st.part_sum + ((size_t)s * st.nparts * kMaxK + j) * 8 + t;
    float sum = 0.0f;
    constexpr int B = 128;  // two memory round trips for the 245 parts of a million rows
    const int np = st.nparts;
    for (int p = 0; p < np; p += B) {
        float v[B];
#pragma unroll
        for (int u = 0; u < B; ++u) v[u] = ps[(size_t)(p + u < np ? p + u : np - 1) * kMaxK * 8];
#pragma unroll
        for (int u = 0; u < B; ++u)
            if (p + u < np) sum = sum + v[u];
    }
    big_sum[((size_t)s * kMaxK + j) * 8 + t] = sum;
}

// The end of an update and the start of the next assignment pass, one workgroup per column block
// (8-float blocks, streaming path, matrix-core assignment).  Thread j makes centroid j — the mean
// of a small cluster from its leaf or of a large one from k_lbg_fold8's sum, the re-seed row of
// an empty cluster (src/vector.rs:315-316, src/utils.rs:98-101) — thread 0 does the loop
// control of src/utils.rs:57,104-106, and all of them the tables of k_assign_mfma8 from the
// centroids they hold.  Needs x 16-byte aligned, ld % 4 == 0 (as the streaming kernel does).
static __global__ void __launch_bounds__(256) k_lbg_finalize_prep8(
    LbgState st, const float *__restrict__ x, int64_t ld, int k, const uint32_t *__restrict__ reseed, int n_reseed,
    float *__restrict__ cb, const float *__restrict__ big_sum, int nb, u32x4 *__restrict__ atab,
    float *__restrict__ aux, uint32_t *__restrict__ stat, uint32_t *__restrict__ stat_next) {
    const int s = blockIdx.x, j = threadIdx.x;
    if (s == 0 && j < kStatSlots) stat[j * kStatStride] = stat_next[j * kStatStride] = 0u;
    if (st.done[s]) return;  // the same in the whole workgroup; a finished block is skipped by the assignment
    float c[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
    if (j < k) {
        const size_t sj = (size_t)s * kMaxK + j;
        const uint32_t cnt = st.count[sj];
        float4 *out = reinterpret_cast<float4 *>(cb + ((size_t)s * k + j) * 8);
        float4 lo4, hi4;
        bool write = true;
        if (cnt == 0) {
            const int pos = st.ubase[s] + (int)st.empty_rank[sj];
            if (pos >= n_reseed) {
                st.err[0] = 1;
                lo4 = out[0];  // the centroid stays
                hi4 = out[1];
                write = false;
            } else {
                const float4 *row =
                    reinterpret_cast<const float4 *>(x + (int64_t)reseed[(size_t)s * n_reseed + pos] * ld + (int64_t)s * 8);
                lo4 = row[0];
                hi4 = row[1];
            }
        } else {
            const float4 *ls = reinterpret_cast<const float4 *>(
                cnt <= (uint32_t)kSeqMax ? st.leaf_sum + ((size_t)s * st.leaf_cap + st.leaf_start[sj]) * 8
                                         : big_sum + ((size_t)s * kMaxK + j) * 8);
            const float d = __uint2float_rn(cnt);
            const float4 a = ls[0], b = ls[1];
            lo4 = make_float4(a.x / d, a.y / d, a.z / d, a.w / d);
            hi4 = make_float4(b.x / d, b.y / d, b.z / d, b.w / d);
        }
        if (write) {
            out[0] = lo4;
            out[1] = hi4;
        }
        c[0] = lo4.x, c[1] = lo4.y, c[2] = lo4.z, c[3] = lo4.w;
        c[4] = hi4.x, c[5] = hi4.y, c[6] = hi4.z, c[7] = hi4.w;
    }
    __syncthreads();  // every thread has read done[s]
    if (j == 0) {
        st.iters[s] += 1;
        if (!st.changed[s]) st.done[s] = 1;
        st.changed[s] = 0;
    }
    mfma8_prep_block(c, s, j, k, nb, atab, aux);
}

}  // namespace vq

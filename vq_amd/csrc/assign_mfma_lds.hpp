// Nearest-centroid assignment with the operands of a whole column block in LDS: blocks of 8 floats with 257 to 2048
// centroids (16-bit codes), blocks of 16 floats with up to 1024.  The scores, their bound and the decision are those of
// k_assign_mfma8 (assign_mfma.hpp); what differs is where the operands lie and how a row's best centroids are kept.
//
// This translation unit must be compiled with -ffp-contract=off.
#pragma once
#include "assign_mfma.hpp"

namespace vq {

constexpr int kBig8Max = 2048, kLds16Max = 1024;
// Components of the padding centroids: +inf, so that their distance to every finite row is +inf wherever the block's
// centroids lie (a scale bounds their spread, not their place).  In a pick they are never clear of a centroid whose
// distance is finite, and beside one that overflows they tie, which the reference's distances of j < k decide.
constexpr float kLdsFar = __builtin_inff();
constexpr float kBig8Rms = 1e30f;   // largest mean square norm about the centre that is scored

enum { CODES_LBG = 0, CODES_U8 = 1, CODES_U16 = 2 };  // [m][n] bytes in place (old -> new), [n][m] bytes, [n][m] 16 bits
struct LdsArgs {
    AssignArgs a;          // 16-byte aligned codebooks; codes: see above (CODES_U16: codes16)
    uint16_t *codes16;
    int64_t stride;        // workgroups of a column block
    uint32_t *stat, *stat_next;  // counters of undecided pairs: of this pass, and of the next (cleared)
};

// Centroids padded to whole pairs of blocks of 32; the operand (4 bytes per float) and the centroid itself, under
// cosine its norm and the reciprocal.
inline int lds_padded(int k) { return (k + 63) / 64 * 64; }
inline size_t assign_lds(bool cosine, int k, int sd) { return (size_t)lds_padded(k) * (8 * sd + (cosine ? 8 : 0)); }

// The workgroup's copy of its block's centroids: planes of four dimensions as in Lds8, runs of 64 bytes with the order
// inside a run depending on the run, so that a phase of the pick's reads, sixteen runs at random, meets all banks.
// A lane half's dimensions are SD / 8 planes side by side.
template <int SD> struct LdsBlock {
    static constexpr int NH = SD / 2, Q = SD / 8;  // dimensions and planes of a half
    char *cl;
    int plane;
    __device__ __forceinline__ int run(int j, int h) const { return h * Q * plane + j * 16 + ((j >> 4) & 3) * 16; }
    __device__ __forceinline__ float4 at(int run, int i, int q) const {
        return *reinterpret_cast<const float4 *>(cl + (run ^ (i * 16)) + q * plane);
    }
    __device__ __forceinline__ void piece(int run, int i, float (&c)[NH]) const {
#pragma unroll
        for (int q = 0; q < Q; ++q) {
            const float4 v = at(run, i, q);
            c[4 * q] = v.x, c[4 * q + 1] = v.y, c[4 * q + 2] = v.z, c[4 * q + 3] = v.w;
        }
    }
    __device__ __forceinline__ void set(int j, int piece16, float4 v) const {  // the centroid's 16-byte piece
        *reinterpret_cast<float4 *>(cl + (run(j & ~3, 0) ^ ((j & 3) * 16)) + piece16 * plane) = v;
    }
    __device__ __forceinline__ float component(int j, int t) const {
        return *reinterpret_cast<const float *>(cl + (run(j & ~3, 0) ^ ((j & 3) * 16)) + (t >> 2) * plane + (t & 3) * 4);
    }
    __device__ __forceinline__ void load(int j, float (&c)[SD]) const {
        const int r = run(j & ~3, 0);
#pragma unroll
        for (int q = 0; q < 2 * Q; ++q) {
            const float4 v = at(r, j & 3, q);
            c[4 * q] = v.x, c[4 * q + 1] = v.y, c[4 * q + 2] = v.z, c[4 * q + 3] = v.w;
        }
    }
};

// The undecided rows of a tile, one after the other: a lane takes the centroids lane, lane + 64, ... by fused
// sums and keeps the two smallest.  One lane with one centroid within 2^-16 of the smallest has the answer;
// otherwise the reference's distances decide, the first of the smallest (a NaN sorts behind +inf, centroid 0 wins
// where it is NaN or nothing is below +inf).
template <int METRIC, int SD>
__device__ __forceinline__ int exact_rows_lds(unsigned long long todo, int code, const LdsBlock<SD> &cl, const float *norms,
                                              int kp, const float (&xr)[SD], float rx, int k, int lane) {
    constexpr uint32_t kInfKey = METRIC == M_COS ? 0xff800000u : 0x7f800000u;  // sort key of +inf
    constexpr int M = METRIC == M_COS ? M_COS : M_SQ;  // Euclidean: squares first
    const int at0 = cl.run(lane & ~3, 0) ^ ((lane & 3) * 16);  // of centroid lane; 64 centroids on is 1 KB on
    while (todo) {
        const int src = __builtin_amdgcn_readfirstlane(__ffsll(todo) - 1);
        todo &= todo - 1;
        float xs[SD];
#pragma unroll
        for (int d = 0; d < SD; ++d) xs[d] = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(xr[d]), src));
        int best = -1;
        {
            const float rxs = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(rx), src));
            uint32_t lo = 0xffffffffu, second = 0xffffffffu, first = 0;
            int at = 0;
            for (int q = 0; q < k; q += 64) {
                float c[SD];
#pragma unroll
                for (int u = 0; u < SD / 4; ++u) {
                    const float4 v = *reinterpret_cast<const float4 *>(cl.cl + at0 + 16 * q + u * cl.plane);
                    c[4 * u] = v.x, c[4 * u + 1] = v.y, c[4 * u + 2] = v.z, c[4 * u + 3] = v.w;
                }
                float d = share8<METRIC, SD>(xs, c);
                if constexpr (METRIC == M_COS) d = __builtin_fmaf(-(d * rxs), norms[kp + q + lane], 1.001f);
                const uint32_t key = __float_as_uint(d);
                if (q == 0) first = key;
                second = umin_u32(second, key < lo ? lo : key);
                at = key < lo ? q + lane : at;
                lo = umin_u32(lo, key);
            }
            const uint32_t least = wave_umin(lo);
            const float b = __uint_as_float(least);
            const uint32_t close = __float_as_uint(METRIC == M_COS ? b + 1.1444091796875e-05f : __builtin_fmaf(b, 1.0000152587890625f, 1e-36f));
            const unsigned long long who = __ballot(lo <= close), also = __ballot(second <= close);
            const int j = __builtin_amdgcn_readlane(at, __ffsll(who | 1ull << 63) - 1);
            const uint32_t d0 = (uint32_t)__builtin_amdgcn_readlane((int)first, 0);
            // (below 1e34: no sum near overflow; centroid 0 is a number; not one of the padding)
            if (least < 0x77f684dfu && d0 <= 0x7f800000u && __popcll(who) == 1 && !also && j < k) best = j;
        }
        if (best < 0) {  // uniform
            const float na = METRIC == M_COS ? seq_norm8(xs) : 0.0f;
            auto key_of = [&](int j) {
                float c[SD];
                cl.load(j, c);
                const float d = dist8<M>(xs, c, na, METRIC == M_COS ? norms[j] : 0.0f);
                return j < k && d == d ? dist_key<M>(d) : 0xffffffffu;
            };
            uint32_t lo = 0xffffffffu;
            for (int q = 0; q < k; q += 64) lo = umin_u32(lo, key_of(q + lane));
            const uint32_t best_key = wave_umin(lo);
            uint32_t close = best_key;  // keys up to here may be the smallest distance
            float root = 0.0f;
            if constexpr (METRIC == M_EUCLID) {
                const float b = __uint_as_float(best_key);
                close = __float_as_uint(__builtin_fmaf(b, 4.76837158203125e-07f, b));
                root = sqrtf(b);
            }
            best = 0;
            const bool nan0 = __builtin_amdgcn_readlane((int)key_of(lane), 0) == -1;  // centroid 0's
            for (int q = 0; q < k && !nan0 && best_key < kInfKey; q += 64) {
                const uint32_t key = key_of(q + lane);
                const bool is = METRIC == M_EUCLID ? key <= close && sqrtf(__uint_as_float(key)) == root : key == close;
                const unsigned long long f = __ballot(is);
                if (f) {
                    best = q + __ffsll(f) - 1;
                    break;
                }
            }
        }
        code = lane == src ? best : code;
    }
    return code;
}

// One workgroup = one column block: its operands (1 KB per 32 centroids) and centroids lie in LDS, made by the
// workgroup itself, and its waves walk over tiles of 32 rows on their own, no barrier after the set-up.  The
// 32 scores that a lane has of 64 centroids go into four sets of eight, {32 b + 8 p + 4 h + 0..3} of two neighbouring
// blocks b: 16 minima, four tags and five operations for the two smallest keys, 25 instructions where sets of
// four take 34.  FOUR: sets of four, the runs themselves, where there are at most four pairs of blocks and the pick
// among eight centroids of 16 floats is more than that saves (eight -> four, Euclidean: 600,000 rows x 8 blocks, k = 256
// 195 -> 181 us, 60,000 x 10 38.4 -> 34.0, k = 64 28.9 -> 24.2, 10,000 x 10 18.5 -> 15.5).
// Even and odd pairs of blocks, and the two lane halves, each have two smallest keys of their own, so that the four
// best sets are known with their tags and a row that only two sets can win is decided among their sixteen
// centroids; the others, a tenth of the pairs that one bound leaves open, go through all k.
// The matrix instructions of the next 64 centroids issue between the halves of this selection.
// Against chunks of 256 centroids, each with its own pass over the rows, and a merge, 16 blocks, Euclidean: 300,000 rows,
// k = 300 240 -> 140 us, 512 269 -> 170, 1024 515 -> 235; 200,000, k = 1500 568 -> 249; 150,000, k = 2048 613 -> 243;
// 1,000, k = 257 20 -> 11, k = 2048 84 -> 30; 100,000 x 12 blocks of 7, k = 1024 269 -> 93.  Bound by vector-instruction
// issue (26 per 64 centroids and tile) and the matrix instructions that only partly hide behind it.
// LBG: codes in place, changed[s] set where one differs, converged blocks left out.
template <int METRIC, int SD, int CODES>
__global__ void __launch_bounds__(SD == 8 ? 1024 : 768, SD == 8 ? 4 : 3) k_assign_mfma_lds(LdsArgs args) {
    extern __shared__ __attribute__((aligned(16))) char lds_block[];
    __shared__ float red[2][16][SD], mu_all[SD];
    constexpr bool COS = METRIC == M_COS, LBG = CODES == CODES_LBG;
    constexpr int NH = SD / 2, NI = SD / 8;  // dimensions of a lane half, matrix instructions per 32 centroids
    constexpr bool FOUR = SD == 16 && CODES != CODES_U16;  // sets of four (up to 256 centroids)
    const AssignArgs &a = args.a;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const int T = (int)blockDim.x, W = T >> 6;
    const int r = lane & 31, h = lane >> 5;
    const int m = a.m, k = a.k, kp = (k + 63) / 64 * 64, np = kp / 64;
    // (blocks to XCDs as in k_assign_mfma8: the column blocks of the same rows on one XCD)
    const unsigned per_chunk = 8u * (unsigned)m;
    const unsigned chunk_id = blockIdx.x / per_chunk, rem = blockIdx.x % per_chunk;
    const int s = (int)(rem / 8u);
    const int64_t first_wg = (int64_t)chunk_id * 8 + (rem % 8u);
    const int64_t ntiles = (a.n + 31) / 32;
    if (first_wg * W >= ntiles) return;
    if (blockIdx.x == 0)
        for (int i = threadIdx.x; i < kStatSlots; i += T) args.stat_next[i * kStatStride] = 0u;
    if constexpr (LBG) {
        if (block_done(a, s)) return;  // uniform
    }

    u32x4 *at = reinterpret_cast<u32x4 *>(lds_block);  // [kp / 32][NI][64]
    const LdsBlock<SD> cl{lds_block + kp * 4 * SD, kp * 16};
    float *norms = reinterpret_cast<float *>(lds_block + kp * 8 * SD);
    {
        constexpr int P = SD / 4;  // 16-byte pieces of a centroid
        const float4 *src = reinterpret_cast<const float4 *>(a.cb + (size_t)s * k * SD);
        for (int i = threadIdx.x; i < P * kp; i += T)
            cl.set(i / P, i % P, i < P * k ? src[i] : make_float4(kLdsFar, kLdsFar, kLdsFar, kLdsFar));
    }
    __syncthreads();
    float mu[SD], sg = kCosScale, bad = 0.0f;
    if constexpr (COS) {
        for (int j = threadIdx.x; j < kp; j += T) {
            float c[SD];
            cl.load(j, c);
            const float nc = seq_norm8(c);
            norms[j] = nc;
            norms[kp + j] = nc == 0.0f || j >= k ? 0.0f : 1.0f / nc;
        }
#pragma unroll
        for (int t = 0; t < SD; ++t) mu[t] = 0.0f;
    } else {
        // a thread per dimension and share of the centroids: two or three shuffles where a sum of all dimensions in
        // every thread took six for each (1,000 rows x 10 blocks of 16: 17.7 -> 10.8 us)
        const int t = threadIdx.x % SD, G = T / SD;
        float v = 0.0f;
        for (int j = threadIdx.x / SD; j < k; j += G) v += cl.component(j, t) * 0.00048828125f;  // / 2048: no overflow
#pragma unroll
        for (int off = SD; off < 64; off <<= 1) v += __shfl_xor(v, off);
        if (lane < SD) red[0][wave][t] = v;
        __syncthreads();
        v = 0.0f;
        for (int w = 0; w < W; ++w) v += red[0][w][t];
        v *= 2048.0f / (float)k;
        if ((int)threadIdx.x < SD) mu_all[t] = v;
        float p = 0.0f;
        for (int j = threadIdx.x / SD; j < k; j += G) {
            const float d = (cl.component(j, t) - v) * 0.015625f;
            p = __builtin_fmaf(d, d, p);  // / 4096
        }
#pragma unroll
        for (int off = 32; off > 0; off >>= 1) p += __shfl_xor(p, off);
        if (lane == 0) red[1][wave][0] = p;
        __syncthreads();
#pragma unroll
        for (int u = 0; u < SD; ++u) mu[u] = mu_all[u];
        float r2 = 0.0f;
        for (int w = 0; w < W; ++w) r2 += red[1][w][0];
        sg = mfma8_scale(r2 * (4096.0f / (float)k), 1, kBig8Rms);  // root mean square 2 ... 4: none longer than 181
        bad = sg - sg;
    }
    float mc2 = 0.0f, mdc = 0.0f;
    for (int j = threadIdx.x; j < kp; j += T) {
        float c[SD];
        cl.load(j, c);
        const bool live = j < k;
        const float nc = COS && live ? norms[j] : 1.0f;
        HalfOp<NH> o[2];
#pragma unroll
        for (int hh = 0; hh < 2; ++hh) {
            float v[NH];
#pragma unroll
            for (int t = 0; t < NH; ++t) {
                const float e = c[NH * hh + t];
                v[t] = !live ? 0.0f : COS ? (nc == 0.0f ? 0.0f : -2.0f * (e * (1.0f / nc)) * kCosScale) : -2.0f * ((e - mu[NH * hh + t]) * sg);
            }
            o[hh] = half_op<NH>(v);
        }
        const float c2 = COS && nc == 0.0f ? kCosScale * kCosScale : o[0].n2 + o[1].n2;
        if (live) {
            float x = c2 + bad;
            if (COS && !(nc == 0.0f || (nc >= 1e-15f && nc <= 1e15f))) x = __builtin_nanf("");
            mc2 = (mc2 == mc2 && x == x) ? fmaxf(mc2, x) : __builtin_nanf("");
            mdc = fmaxf(mdc, o[0].d2 + o[1].d2);
        }
#pragma unroll
        for (int hh = 0; hh < 2; ++hh) {
            uint32_t w[NH];
#pragma unroll
            for (int t = 0; t < NH - 1; ++t) w[t] = o[hh].w[t];
            w[NH - 1] = c2_word(c2, hh, live);
#pragma unroll
            for (int i = 0; i < NI; ++i)
                at[((j / 32) * NI + i) * 64 + 32 * hh + j % 32] = u32x4{w[4 * i], w[4 * i + 1], w[4 * i + 2], w[4 * i + 3]};
        }
    }
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) {
        const float o = __shfl_xor(mc2, off);
        mc2 = (mc2 == mc2 && o == o) ? fmaxf(mc2, o) : __builtin_nanf("");
        mdc = fmaxf(mdc, __shfl_xor(mdc, off));
    }
    if (lane == 0) {
        red[0][wave][0] = mc2;
        red[0][wave][1] = mdc;
    }
    __syncthreads();  // (red[0] was read before the barrier that red[1] needed)
    for (int w = 0; w < W; ++w) {
        const float o = red[0][w][0];
        mc2 = (mc2 == mc2 && o == o) ? fmaxf(mc2, o) : __builtin_nanf("");
        mdc = fmaxf(mdc, red[0][w][1]);
    }
    float muh[NH];
#pragma unroll
    for (int u = 0; u < NH; ++u) muh[u] = COS ? 0.0f : -((h ? mu[NH + u] : mu[u]) * sg);
    const uint32_t keep = opaque_vgpr(0xFFFFFF00u);
    const float acc8 = NH / 4 * 4.57763671875e-05f * mc2;  // see decided8

    // tiles t, t + step, ...; rows two tiles ahead
    const int64_t step = args.stride * W;
    int64_t t = first_wg * W + wave;
    const uint32_t loff = 4u * ((uint32_t)r * (uint32_t)a.ld + (uint32_t)NH * (uint32_t)h);
    typedef float rowpiece __attribute__((ext_vector_type(4), aligned(4)));
    auto fetch = [&](int64_t tile, rowpiece(&v)[NH / 4]) {
        const int64_t row0 = (tile < ntiles ? tile : ntiles - 1) * 32;  // uniform
        const char *base = reinterpret_cast<const char *>(a.x + row0 * a.ld + (int64_t)s * SD);
        const uint32_t o = r < a.n - row0 ? loff : 4u * NH * (uint32_t)h;
#pragma unroll
        for (int q = 0; q < NH / 4; ++q) v[q] = *reinterpret_cast<const rowpiece *>(base + o + 16 * q);
    };
    uint8_t oa = 0, ob = 0;
    auto fetch_c = [&](int64_t tile) {
        const int64_t row0 = (tile < ntiles ? tile : ntiles - 1) * 32;
        return a.codes[(size_t)s * a.n + row0 + (r < a.n - row0 ? r : 0)];
    };
    uint32_t n_exact = 0;
    bool chg = false;
    rowpiece xa[NH / 4], xb[NH / 4];
    fetch(t, xa);
    if constexpr (LBG) oa = fetch_c(t);
    fetch(t + step, xb);
    if constexpr (LBG) ob = fetch_c(t + step);
    for (; t < ntiles; t += step) {
        float xraw[NH];
#pragma unroll
        for (int u = 0; u < NH; ++u) xraw[u] = xa[u / 4][u % 4];
#pragma unroll
        for (int q = 0; q < NH / 4; ++q) xa[q] = xb[q];
        fetch(t + 2 * step, xb);
        const uint8_t old = oa;
        oa = ob;
        if constexpr (LBG) ob = fetch_c(t + 2 * step);
        const RowOp<NH> row = row_op<METRIC, NH>(xraw, sg, muh);
        const floatx16 zero = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
        int m1 = 0x7f800000, m2 = 0x7f800000, o1 = 0x7f800000, o2 = 0x7f800000;  // +inf; even and odd pairs
        floatx16 p0, p1, q0, q1;
#define VQ_MFMA(av, xv, from, acc)                                                                                    \
    acc = __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(f16x8, av), __builtin_bit_cast(f16x8, xv), from, 0, 0, 0);
#define VQ_MIN8(c, d, p)                                                                                              \
    imin(imin(imin(imin(imin(imin(imin(__float_as_int(c[4 * p]), __float_as_int(c[4 * p + 1])),                       \
                                   __float_as_int(c[4 * p + 2])), __float_as_int(c[4 * p + 3])),                      \
                        __float_as_int(d[4 * p])), __float_as_int(d[4 * p + 1])), __float_as_int(d[4 * p + 2])),      \
         __float_as_int(d[4 * p + 3]))
#define VQ_MIN4(c, p)                                                                                                 \
    imin(imin(imin(__float_as_int(c[4 * p]), __float_as_int(c[4 * p + 1])), __float_as_int(c[4 * p + 2])),            \
         __float_as_int(c[4 * p + 3]))
#define VQ_KEY4(c, p, tag) (int)(((uint32_t)VQ_MIN4(c, p) & keep) | (tag))
#define VQ_KEY(c, d, p, tag) key[p] = (int)(((uint32_t)VQ_MIN8(c, d, p) & keep) | (tag));
        // selection of 64 centroids (scores in c, d) with the matrix instructions of the next 64 (into e, f)
#define VQ_PAIR(c, d, e, f, first, second, T0, T1, T2, T3, T4, T5, T6, T7, next)                                      \
    {                                                                                                                 \
        int key[4];                                                                                                   \
        VQ_MFMA(n0[0], row.b16[0], zero, e)                                                                           \
        if constexpr (NI == 2) VQ_MFMA(n1[0], row.b16[0], zero, f)                                                    \
        __builtin_amdgcn_sched_barrier(0);                                                                            \
        if constexpr (FOUR) {                                                                                         \
            top2_push4(first, second, VQ_KEY4(c, 0, T0), VQ_KEY4(c, 1, T1), VQ_KEY4(c, 2, T2), VQ_KEY4(c, 3, T3));    \
        } else {                                                                                                      \
            VQ_KEY(c, d, 0, T0) VQ_KEY(c, d, 1, T1)                                                                   \
        }                                                                                                             \
        __builtin_amdgcn_sched_barrier(0);                                                                            \
        if constexpr (NI == 2) {                                                                                      \
            VQ_MFMA(n0[NI - 1], row.b16[NI - 1], e, e)                                                                \
            VQ_MFMA(n1[NI - 1], row.b16[NI - 1], f, f)                                                                \
        } else {                                                                                                      \
            VQ_MFMA(n1[0], row.b16[0], zero, f)                                                                       \
        }                                                                                                             \
        operands(next);                                                                                               \
        __builtin_amdgcn_sched_barrier(0);                                                                            \
        if constexpr (FOUR) {                                                                                         \
            top2_push4(first, second, VQ_KEY4(d, 0, T4), VQ_KEY4(d, 1, T5), VQ_KEY4(d, 2, T6), VQ_KEY4(d, 3, T7));    \
        } else {                                                                                                      \
            VQ_KEY(c, d, 2, T2) VQ_KEY(c, d, 3, T3)                                                                   \
            top2_push4(first, second, key[0], key[1], key[2], key[3]);                                                \
        }                                                                                                             \
        __builtin_amdgcn_sched_barrier(0);                                                                            \
    }
        // the tags of the sets, one scalar register each: tag = 8 * pair + 2 * set (FOUR: 16 * pair + 2 * set)
        uint32_t t0 = 0, t1 = 2, t2 = 4, t3 = 6, t4 = 8, t5 = 10, t6 = 12, t7 = 14;
        uint32_t u0 = 16, u1 = 18, u2 = 20, u3 = 22, u4 = 24, u5 = 26, u6 = 28, u7 = 30;  // FOUR, odd pairs
        auto opaque = [](uint32_t &v) { asm volatile("" : "+s"(v)); };  // (else each is made again from one of them)
        const u32x4 *ap = at + lane;
        u32x4 n0[NI], n1[NI];  // of the next pair's two blocks
        auto operands = [&](int pair) {
#pragma unroll
            for (int i = 0; i < NI; ++i) {
                n0[i] = ap[(pair * 2 * NI + i) * 64];
                n1[i] = ap[((pair * 2 + 1) * NI + i) * 64];
            }
        };
        operands(0);
        VQ_MFMA(n0[0], row.b16[0], zero, p0)
        VQ_MFMA(n1[0], row.b16[0], zero, p1)
        if constexpr (NI == 2) {
            VQ_MFMA(n0[NI - 1], row.b16[NI - 1], p0, p0)
            VQ_MFMA(n1[NI - 1], row.b16[NI - 1], p1, p1)
        }
        operands(np > 1 ? 1 : 0);
        for (int p = 0; p < np; p += 2) {
            opaque(t0), opaque(t1), opaque(t2), opaque(t3), opaque(t4), opaque(t5), opaque(t6), opaque(t7);
            if constexpr (FOUR) {
                opaque(u0), opaque(u1), opaque(u2), opaque(u3), opaque(u4), opaque(u5), opaque(u6), opaque(u7);
                VQ_PAIR(p0, p1, q0, q1, m1, m2, t0, t1, t2, t3, t4, t5, t6, t7, p + 2 < np ? p + 2 : 0)
                if (p + 1 < np) VQ_PAIR(q0, q1, p0, p1, o1, o2, u0, u1, u2, u3, u4, u5, u6, u7, p + 3 < np ? p + 3 : 0)
                t0 += 32, t1 += 32, t2 += 32, t3 += 32, t4 += 32, t5 += 32, t6 += 32, t7 += 32;
                u0 += 32, u1 += 32, u2 += 32, u3 += 32, u4 += 32, u5 += 32, u6 += 32, u7 += 32;
            } else {
                VQ_PAIR(p0, p1, q0, q1, m1, m2, t0, t1, t2, t3, 0, 0, 0, 0, p + 2 < np ? p + 2 : 0)
                if (p + 1 < np) VQ_PAIR(q0, q1, p0, p1, o1, o2, t4, t5, t6, t7, 0, 0, 0, 0, p + 3 < np ? p + 3 : 0)
                t0 += 16, t1 += 16, t2 += 16, t3 += 16, t4 += 16, t5 += 16, t6 += 16, t7 += 16;
            }
        }
#undef VQ_MFMA
#undef VQ_MIN8
#undef VQ_MIN4
#undef VQ_KEY4
#undef VQ_KEY
#undef VQ_PAIR
        m1 |= h;  // bit 0 of the tag: the lane half
        o1 |= h;
        int f0, f1, g0, g1, e0, e1;
        swap_halves(m1, f0, f1);
        swap_halves(o1, g0, g1);
        swap_halves(imin(m2, o2), e0, e1);
        const int lo_a = imin(f0, f1), hi_a = imax(f0, f1), lo_b = imin(g0, g1), hi_b = imax(g0, g1);
        const int mid_a = imax(lo_a, lo_b), mid_b = imin(hi_a, hi_b);
        const int set1 = imin(lo_a, lo_b), set2 = imin(mid_a, mid_b);        // the two best sets with a tag
        const int others = imin(imax(mid_a, mid_b), imin(e0, e1));           // no other set is below
        const float s1 = __int_as_float(set1), s2 = __int_as_float(imin(set2, others));
        const int64_t row0 = t * 32;
        const bool mine = h == 0 && r < a.n - row0;  // the lane's row exists
        bool near = decided8<METRIC, NH>(s1, s2, row, mdc, acc8);
        // The best of a set's eight centroids, runs first and first + 32: each lane half sums its four dimensions of
        // all of them, the lower half then holds the first run's distances, the upper half the second's, the place in
        // the run in the two low bits.  at: the best; lo, hi: the two smallest keys (lower lanes).
        auto first_of = [](int set) {
            const uint32_t tag = (uint32_t)set & 0xFFu;
            if constexpr (FOUR) return (int)((tag >> 3) * 32 + ((tag >> 1) & 3u) * 8 + (tag & 1u) * 4);
            return (int)((tag >> 3) * 64 + ((tag >> 1) & 3u) * 8 + (tag & 1u) * 4);
        };
        // FOUR: the one run of a set, its first two centroids in the lower half, the others in the upper.
        auto pick = [&](int first, int &at, int &lo, int &hi) {
            if constexpr (FOUR) {
                const int ra = cl.run(first, h), j0 = first + 2 * h;
                float2 inv = make_float2(0.f, 0.f);
                if constexpr (COS) inv = *reinterpret_cast<const float2 *>(norms + kp + j0);
                int ky[2];
#pragma unroll
                for (int i = 0; i < 2; ++i) {
                    float ca[NH], cb[NH];
                    cl.piece(ra, i, ca);
                    cl.piece(ra, i + 2, cb);
                    const auto sw = __builtin_amdgcn_permlane32_swap(__float_as_int(share8<METRIC, NH>(xraw, ca)),
                                                                     __float_as_int(share8<METRIC, NH>(xraw, cb)), false, false);
                    float d = __int_as_float((int)sw[0]) + __int_as_float((int)sw[1]);
                    if constexpr (COS) d = j0 + i < k ? __builtin_fmaf(-(d * row.rx), i ? inv.y : inv.x, 1.001f) : 1e30f;
                    ky[i] = (int)((__float_as_uint(d) & 0xFFFFFFFCu) | (uint32_t)(i + 2 * h));
                }
                int l0, l1, h0, h1;
                swap_halves(imin(ky[0], ky[1]), l0, l1);
                swap_halves(imax(ky[0], ky[1]), h0, h1);
                lo = imin(l0, l1);
                hi = imin3(imax(l0, l1), h0, h1);
                at = first + (lo & 3);
                return;
            }
            const int ra = cl.run(first, h), rb = cl.run(first + 32, h);
            const int j0 = first + 32 * h;
            float4 inv = make_float4(0.f, 0.f, 0.f, 0.f);
            if constexpr (COS) inv = *reinterpret_cast<const float4 *>(norms + kp + j0);
            const float iv[4] = {inv.x, inv.y, inv.z, inv.w};
            int ky[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                float ca[NH], cb[NH];
                cl.piece(ra, i, ca);
                cl.piece(rb, i, cb);
                const auto sw = __builtin_amdgcn_permlane32_swap(__float_as_int(share8<METRIC, NH>(xraw, ca)),
                                                                 __float_as_int(share8<METRIC, NH>(xraw, cb)), false, false);
                float d = __int_as_float((int)sw[0]) + __int_as_float((int)sw[1]);
                if constexpr (COS) d = j0 + i < k ? __builtin_fmaf(-(d * row.rx), iv[i], 1.001f) : 1e30f;
                ky[i] = (int)((__float_as_uint(d) & 0xFFFFFFFCu) | (uint32_t)i);
            }
            const int a3 = imin3(ky[0], ky[1], ky[2]), b3 = imed3a(ky[0], ky[1], ky[2]);
            int l0, l1, h0, h1;
            swap_halves(imin(a3, ky[3]), l0, l1);
            swap_halves(imin(b3, imax(a3, ky[3])), h0, h1);
            lo = imin(l0, l1);
            hi = imin3(imax(l0, l1), h0, h1);
            at = first + (l1 < l0 ? 32 : 0) + (lo & 3);  // (lower half: 0 its own, 1 the partner's)
        };
        // (2^-16: the sums' rounding and the reference's, the bits left out; 1e-36: subnormal sums of squares)
        auto apart = [](int lo, int hi) {
            const float best = __int_as_float(lo & ~3), second = __int_as_float(hi & ~3);
            return COS ? second - best > 1.1444091796875e-05f : __builtin_fmaf(second, 0.9999847412109375f, -1e-36f) > best;
        };
        const int first = first_of(set1);
        int code, lo, hi;
        pick(first, code, lo, hi);
        bool clear = apart(lo, hi);
        int other = -1;  // the second set, where it may have the answer
        unsigned long long todo = __ballot(mine && !near);
        if (todo) {  // the same in every lane
            if (!near && decided8<METRIC, NH>(s1, __int_as_float(others), row, mdc, acc8)) other = first_of(set2);
            const bool two = other >= 0;
            if (__ballot(mine && two)) {
                int code2, lo2, hi2;
                pick(two ? other : first, code2, lo2, hi2);
                if (two) {
                    code = lo2 < lo ? code2 : code;
                    hi = imin3(imax(lo, lo2), hi, hi2);
                    lo = imin(lo, lo2);
                    clear = apart(lo, hi);
                    near = true;
                }
                todo = __ballot(mine && !near);
            }
        }
        const unsigned long long ties = __ballot(mine && near && !clear);
        if (todo | ties) {  // the same in every lane
            float xs[SD];  // the lane's row
#pragma unroll
            for (int u = 0; u < NH; ++u) {
                int xl, xh;
                swap_halves(__float_as_int(xraw[u]), xl, xh);
                xs[u] = __int_as_float(xl);
                xs[NH + u] = __int_as_float(xh);
            }
            if (ties) {  // the sets' centroids by the reference's distances: the first of the smallest
                const float na = COS ? seq_norm8(xs) : 0.0f;
                float bd = 0.0f;
                int bj = -1;
                constexpr int N = FOUR ? 4 : 8;  // centroids of a set
                for (int i = 0; i < (__ballot(other >= 0 && !clear) ? 2 * N : N); ++i) {
                    const int j = (i < N || other < 0 ? first : other) + (i & 3) + (FOUR ? 0 : ((i >> 2) & 1) * 32);
                    float c[SD];
                    cl.load(j, c);
                    const float d = dist8<METRIC>(xs, c, na, COS ? norms[j] : 0.0f);
                    if (j < k && (bj < 0 || d < bd || (d == bd && j < bj))) {
                        bd = d;
                        bj = j;
                    }
                }
                code = clear ? code : bj;
            }
            if (todo) {
                n_exact += (uint32_t)__popcll(todo);
                code = exact_rows_lds<METRIC, SD>(todo, code, cl, norms, kp, xs, row.rx, k, lane);
            }
        }
        if (mine) {
            if constexpr (CODES == CODES_U16) {
                args.codes16[(size_t)(row0 + r) * m + s] = (uint16_t)code;
            } else if constexpr (CODES == CODES_U8) {
                a.codes[(size_t)(row0 + r) * m + s] = (uint8_t)code;
            } else if (old != (uint8_t)code) {
                a.codes[(size_t)s * a.n + row0 + r] = (uint8_t)code;
                chg = true;
            }
        }
    }
    if constexpr (LBG) {
        // once per wave, and only where the flag still reads 0 (see k_assign_mfma8)
        if (__any(chg) && lane == 0 && a.changed[s] == 0) a.changed[s] = 1;
    }
    if (lane == 0 && n_exact)
        atomicAdd(args.stat + ((first_wg * W + wave) & (kStatSlots - 1)) * kStatStride, n_exact);
}

// One round of workgroups: sixteen waves per compute unit (blocks of 8 floats; twelve with 16), as two workgroups, or
// three, while their LDS leaves room.  Eight workgroups at a time per column block, for the order of the blocks on the XCDs:
// full for m = 8, 16, 32, for others not, and from m = 33 at k = 2048 a little over one round.  Two million pairs,
// Euclidean: k = 2048 m = 16 227 us, 17 (136 of 256 workgroups) 346, 24 256, 32 223, 33 (264) 371, 64 238; k = 1024 235, 270, 288, 243, 381,
// 241; 16 floats, k = 256 m = 16 181 (300,000 rows), 17 207, 24 267, 25 325.
template <int METRIC, int SD, int CODES>
inline hipError_t launch_mfma_lds(hipStream_t stream, LdsArgs &args) {
    const size_t lds = assign_lds(METRIC == M_COS, args.a.k, SD);
    const int waves_cu = SD == 8 ? 16 : 12;
    const int wgs_cu = lds <= 50 * 1024 && SD == 16 ? 3 : lds <= 77 * 1024 ? 2 : 1, waves = waves_cu / wgs_cu;
    const int64_t tiles = (args.a.n + 31) / 32;
    int64_t stride = 256 * wgs_cu / args.a.m / 8 * 8;
    if (stride < 8) stride = 8;
    const int64_t most = ((tiles + waves - 1) / waves + 7) / 8 * 8;
    if (stride > most) stride = most;
    if (stride * args.a.m >= (1LL << 31)) return hipErrorInvalidConfiguration;
    args.stride = stride;
    const void *kern = reinterpret_cast<const void *>(k_assign_mfma_lds<METRIC, SD, CODES>);
    const hipError_t e = hipFuncSetAttribute(kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    if (e != hipSuccess) return e;
    void *kargs[] = {&args};
    return hipLaunchKernel(kern, dim3((unsigned)(stride * args.a.m)), dim3((unsigned)(64 * waves)), kargs, lds, stream);
}

}  // namespace vq

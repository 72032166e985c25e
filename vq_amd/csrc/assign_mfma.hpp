// Nearest-centroid assignment for squared-L2 / Euclidean on the matrix cores, exact by re-check.
//
// The scores  s[j] = ||c_j||^2 + ||x||^2 - 2 x.c_j  of 32 rows against 32 centroids at a time come
// out of the matrix cores.  The matrix form rounds differently from the reference's sequential
// (x-c)^2 sum, so a row is only decided from the scores when its best candidates are further
// apart than a bound on every error involved (operand splitting, matrix accumulation, the index
// bits packed into the 8 low mantissa bits, the reference's own rounding).  Then the smallest
// exact distance provably lies where the scores say.  Every other (row, block) pair — exact ties,
// near ties, sqrt collisions under Euclidean, non-finite values — is decided by the
// reference-order argmin, so the result is bit-identical to the all-VALU path for every input.
// The 8-float kernel keeps the two smallest keys over runs of four consecutive centroids (the
// run's smallest score, tagged with the run's first index) and picks inside the best run by exact
// distances; the wide kernel keeps the three smallest scores, one tag per score.
//
// 8-float column blocks (k_assign_mfma8): one product of binary16 operands per score; the undecided
// rows are resolved inside the same wave.  Wider blocks (k_assign_mfma_wide_bf): operands split into bf16
// parts, or rounded to binary16; the undecided pairs are listed for the exact kernel of assign_exact.hpp.
#pragma once
#include <hip/hip_runtime.h>
#include <hip/hip_fp16.h>
#include <stdint.h>

#include "assign_exact.hpp"

namespace vq {

typedef float floatx16 __attribute__((ext_vector_type(16)));

// Score of the padding centroids that fill the last block of 32; a row whose best score is not
// well below it is decided by the exact path.
constexpr float kPadScore = 1e30f;

// Scores are compared through their bit patterns as signed integers: for non-negative floats
// that is the float order, a slightly negative score (cancellation) still sorts below every
// positive one, and integer min / med3 need no NaN canonicalisation.  Two negative scores sort
// in reverse, which only happens inside the error bound, i.e. for pairs that are re-checked.
__device__ __forceinline__ int imin(int a, int b) { return a < b ? a : b; }
__device__ __forceinline__ int imax(int a, int b) { return a > b ? a : b; }
__device__ __forceinline__ int imed3(int a, int b, int c) {
    return imax(imin(a, b), imin(imax(a, b), c));
}
// v_min3_i32 by name: the compiler otherwise splits the chain of smallest keys into pairs of v_min_i32.
__device__ __forceinline__ int imin3(int a, int b, int c) {
    int r;
    asm("v_min3_i32 %0, %1, %2, %3" : "=v"(r) : "v"(a), "v"(b), "v"(c));
    return r;
}

// (score bits & keep) | tag as one v_and_or_b32 with the tag in a scalar register: keep must be a
// vector register the compiler cannot see through (with a literal mask it emits a v_and with the
// literal and a v_or with the scalar operand, twice the issue time).  Left to the compiler rather
// than written as inline assembly so that it inserts the wait states between a matrix
// instruction and the first read of its result.
__device__ __forceinline__ uint32_t opaque_vgpr(uint32_t value) {
    uint32_t r;
    asm volatile("v_mov_b32 %0, %1" : "=v"(r) : "s"(value));
    return r;
}
__device__ __forceinline__ int pack_tag(float score, uint32_t keep, uint32_t tag) {
    return (int)((__float_as_uint(score) & keep) | tag);
}

// The values of lanes l and l ^ 32 in one vector instruction (v_permlane32_swap: the upper half of
// the first operand and the lower half of the second change places).  Lanes below 32 get
// (own, partner), the others (partner, own): for symmetric uses only.
__device__ __forceinline__ void swap_halves(int v, int &a, int &b) {
    const auto r = __builtin_amdgcn_permlane32_swap(v, v, false, false);
    a = (int)r[0];
    b = (int)r[1];
}

// v_med3_i32 / v_max3_i32 by name, for the same reason.  Not for operands that a matrix instruction
// has just written: the compiler does not count wait states for inline assembly.
__device__ __forceinline__ int imed3a(int a, int b, int c) {
    int r;
    asm("v_med3_i32 %0, %1, %2, %3" : "=v"(r) : "v"(a), "v"(b), "v"(c));
    return r;
}
__device__ __forceinline__ int imax3a(int a, int b, int c) {
    int r;
    asm("v_max3_i32 %0, %1, %2, %3" : "=v"(r) : "v"(a), "v"(b), "v"(c));
    return r;
}

// Four new keys into the running three smallest (m1 <= m2 <= m3): 10 operations.  The smallest
// comes out of two min3 steps; the second is the smallest of m2 and the two medians; the third
// is the smallest of everything else that can still be third: the median of those three, the
// two maxima, and m3.
__device__ __forceinline__ void top3_push4(int &m1, int &m2, int &m3, int k0, int k1, int k2, int k3) {
    const int ta = imed3a(m1, k0, k1), xa = imax3a(m1, k0, k1), a1 = imin3(m1, k0, k1);
    const int tb = imed3a(a1, k2, k3), xb = imax3a(a1, k2, k3);
    m1 = imin3(a1, k2, k3);
    const int md = imed3a(m2, ta, tb);
    m2 = imin3(m2, ta, tb);
    m3 = imin(imin3(m3, xa, xb), md);
}

// Four new keys into the running (smallest, second smallest): 5 operations.
// second smallest of {m1, m2, x, y} with m1 <= m2 is min(m2, med3(m1, x, y)).
__device__ __forceinline__ void top2_push4(int &m1, int &m2, int k0, int k1, int k2, int k3) {
    const int ta = imed3(m1, k0, k1);
    const int a1 = imin3(m1, k0, k1);
    const int tb = imed3(a1, k2, k3);
    m1 = imin3(a1, k2, k3);
    m2 = imin3(m2, ta, tb);
}

// ---------------------------------------------------------------------------------------------
// 8-float column blocks on the binary16 matrix cores (v_mfma_f32_32x32x16_f16), one instruction per 32 rows x
// 32 centroids.
//
// Rows and centroids are taken relative to the block's centre and scaled by a power of two (mfma8_scale).
// The lanes of half h = lane / 32 own dimensions [4h, 4h + 4); with a = -2c the 8 contraction slots of that
// half hold
//     ah . xh  (4 slots)   al . xh  (the half's first two dimensions)   1 . (the half's share of ||x||^2)
//     (||c~||^2 in two parts, the higher in the lower half) . 1
// where xh, ah are the values rounded to binary16 and al what that left of a.  So a lane loads and rounds
// only its own 16 bytes of the row, and the scores are the squared distances between the ROUNDED row x~ and the
// ROUNDED centroids c~ up to the accumulation (the share of ||x||^2, the same in every score of the row, only keeps
// them positive; it is enlarged by kLift8 and rounded itself).
// What that is worth: with ex = x - x~ and ec = c - c~ the distances of two centroids differ by
//     d2^2 - d1^2 >= s2 - s1 - 2 |c~1 - c~2| |ex| - 2 sqrt(s1) |ec1| - 2 sqrt(s2) |ec2| - (second order)
// and |c~1 - c~2| <= sqrt(s1) + sqrt(s2): the first candidate has won when
//     s2 - s1 > 4 (sqrt(s2) + e) e,   e = |ex| + max |ec| <= sqrt(2 (|ex|^2 + max |ec|^2)),
// an error in proportion to the DISTANCE, not to the norms.  |ex|^2 is summed as the row is rounded, max |ec|^2
// made with the tables.  On top of it 2^-16 (||x||^2 + max ||c~||^2) for the accumulation of 16 products, the two
// parts of ||c~||^2 (2^-22) and the rounding of x and c relative to the centre (2^-24), and 2^-14 |second| for the
// packed bits and the reference's own rounding.  Non-finite values, and rows beyond the range of binary16, fail
// the test.
// Measured against two instructions of bf16 parts (ah.xh + ah.xl + al.xh; a margin of 2^-13 (||x||^2 + max
// ||c||^2), 0.07-0.3 % of the pairs undecided where this leaves 0.2-1 %): half the matrix instructions and half
// the operand registers, a fifth fewer vector instructions to make the row's operand.  1M x 128, m = 16, k = 256:
// a pass of a fit 382 -> 295-315 us under the profiler; fit and encode 5.19 -> 4.61 ms; encode of 200,000 x 96
// under cosine 95 -> 83 us (with the undecided rows read from registers, exact_rows8).
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef float floatx2 __attribute__((ext_vector_type(2)));
using f16x8 = _Float16 __attribute__((ext_vector_type(8)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

constexpr float kPad8 = 65504.0f;  // padding centroids: ||c~||^2 = 2 kPad8, longer than any that is scored
constexpr float kLift8 = 1.004f;   // the row's share of ||x||^2 in binary16 is then above its rounded operand's
constexpr float kFlush8 = 3.0e-8f; // eight elements below the normal range of binary16, squared
constexpr float kCosScale = 4.0f;  // cosine: the length of rows and centroids

constexpr int kStatSlots = 64;    // counters of undecided pairs, one 128-byte line apart
constexpr int kStatStride = 32;

constexpr int kMfma8Aux = 12;  // floats per column block beside the operands
// aux[s]: [0, 8) minus the centre times the scale, [8] largest ||c~||^2 (NaN: no row of the block may be
// decided by its scores), [9] largest dc^2, [10] the scale
struct Mfma8Tables {
    const u32x4 *atab;     // [m][nb][64]  A operands, lane order
    const float *aux;      // [m][kMfma8Aux]
    uint32_t *stat;        // [kStatSlots * kStatStride]  pairs decided by the exact path (measurement)
    int nb;                // blocks of 32 centroids, padded to an even number
    uint32_t *stat_next = nullptr;  // (OWN) the counters of the pass after this one, to be cleared
};

// float -> bf16 bits, round to nearest even (NaN stays NaN).
__host__ __device__ __forceinline__ uint32_t bf16_rne_bits(float f) {
    uint32_t u = __builtin_bit_cast(uint32_t, f);
    if ((u & 0x7fffffffu) > 0x7f800000u) return (u >> 16) | 0x40u;
    u += 0x7fffu + ((u >> 16) & 1u);
    return u >> 16;
}
__device__ __forceinline__ float bf16_bits_to_float(uint32_t b) { return __uint_as_float(b << 16); }

// two floats -> packed bf16 pair (lo = first), round to nearest even
__device__ __forceinline__ uint32_t bf16_pack2(float a, float b) {
    floatx2 f = {a, b};
    bf16x2 h = __builtin_convertvector(f, bf16x2);
    return __builtin_bit_cast(uint32_t, h);
}

// ---- cosine -----------------------------------------------------------------------------------
// d = 1 - x.c / (|x| |c|) is half the squared distance of x / |x| and c / |c|: rows and centroids are brought
// to length kCosScale, about the origin, and scored like the others.  What this adds to the bound, in units of
// kCosScale^2: the scaling of the row and of the centroid, below 2^-20; the reference (src/distances.rs:141-151),
// whose sums, product of the norms, quotient and difference from 1 leave d within 14 * 2^-24, 2^-18.2 for two
// candidates; the 2^-16 of both norms covers them.  Rows and centroids whose norm is outside [1e-15, 1e15]
// and not zero, where the reference's products may over- or underflow, and rows of norm zero go to the exact
// argmin (a centroid of norm zero has d = 1: its operand is zero and its ||c~||^2 kCosScale^2, in order).
template <int SD> __device__ __forceinline__ float seq_norm8(const float (&c)[SD]) {
    float acc = 0.0f;
#pragma unroll
    for (int t = 0; t < SD; ++t) {
        const float p = c[t] * c[t];
        acc = acc + p;
    }
    return sqrtf(acc);
}
// c divided by its norm; 0, or NaN if the block must not be scored with this centroid in it.
__device__ __forceinline__ float cos_normalise(float (&c)[8], bool &zero) {
    const float nb = seq_norm8(c);
    zero = nb == 0.0f;
    const float inv = zero ? 0.0f : 1.0f / nb;
#pragma unroll
    for (int t = 0; t < 8; ++t) c[t] *= inv;
    return zero || (nb >= 1e-15f && nb <= 1e15f) ? 0.0f : __builtin_nanf("");
}
// Distances as sort keys: smaller distance, smaller unsigned key.  Squared and plain Euclidean
// distances are non-negative, a cosine distance may be a little below zero.
template <int METRIC> __device__ __forceinline__ uint32_t dist_key(float d) {
    const uint32_t b = __float_as_uint(d);
    if constexpr (METRIC == M_COS) return b ^ ((uint32_t)((int)b >> 31) | 0x80000000u);
    return b;
}
template <int METRIC> __device__ __forceinline__ float key_dist(uint32_t k) {
    if constexpr (METRIC == M_COS) return __uint_as_float(k ^ ((k & 0x80000000u) ? 0x80000000u : 0xffffffffu));
    return __uint_as_float(k);
}
// The distance of a row's SD floats to centroid c, in the reference's order; na, nb: the two norms.
template <int METRIC, int SD>
__device__ __forceinline__ float dist8(const float (&x)[SD], const float (&c)[SD], float na, float nb) {
    if constexpr (METRIC == M_COS) {
        const float dot = d_dot<SD>(x, c);
        const float den = na * nb, q = dot / den;
        return (na == 0.0f || nb == 0.0f) ? 1.0f : 1.0f - q;
    } else {
        const float d = d_sq<SD>(x, c);
        return METRIC == M_EUCLID ? sqrtf(d) : d;
    }
}

// The scale of a column block: the power of two that brings the centroids' root mean square norm about the
// centre to 4 ... 8 (r2: the mean square; NaN where the scores cannot decide).  A centroid is then no longer
// than 128 (k <= 256), and a row's share of ||x||^2 fits binary16 up to 32 ... 64 times that norm.
__device__ __forceinline__ float mfma8_scale(float r2, int up = 2, float most = 1e36f) {
    if (r2 == 0.0f) return 1.0f;  // all centroids are the same
    return r2 > 1e-36f && r2 < most ? ldexpf(1.0f, up - (ilogbf(r2) >> 1)) : __builtin_nanf("");
}
// The A operand of one centroid and one lane half: a[t] = -2 c[t] of the half's NH dimensions, scaled: NH / 2
// words of high parts, then the low parts of the first NH - 2 dimensions, one instruction per 8 slots (the last
// word of the last is c2_word's).  Elements below the normal range of binary16 count as zero, whatever the matrix
// cores make of them.  n2, d2: the half's shares of ||c~||^2 and of ||c - c~||^2.
template <int NH> struct HalfOp {
    uint32_t w[NH - 1];
    float n2, d2;
};
__device__ __forceinline__ float f16_normal(float v) {
    const float r = (float)(_Float16)v;
    return fabsf(r) < 6.103515625e-05f ? 0.0f : r;
}
__device__ __forceinline__ uint32_t f16_pack2(float a, float b) {  // round to nearest even
    using h2 = _Float16 __attribute__((ext_vector_type(2)));
    return __builtin_bit_cast(uint32_t, h2{(_Float16)a, (_Float16)b});
}
template <int NH> __device__ __forceinline__ HalfOp<NH> half_op(const float (&a)[NH]) {
    float hi[NH], lo[NH];
    HalfOp<NH> o;
    o.n2 = o.d2 = 0.0f;
#pragma unroll
    for (int t = 0; t < NH; ++t) {
        hi[t] = f16_normal(a[t]);
        lo[t] = t < NH - 2 ? f16_normal(a[t] - hi[t]) : 0.0f;
        const float d = (a[t] - hi[t]) - lo[t], v = hi[t] + lo[t];
        o.n2 = __builtin_fmaf(0.25f * v, v, o.n2);
        o.d2 = __builtin_fmaf(0.25f * d, d, o.d2);
    }
#pragma unroll
    for (int t = 0; t < NH / 2; ++t) o.w[t] = f16_pack2(hi[2 * t], hi[2 * t + 1]);
#pragma unroll
    for (int t = 0; t < NH / 2 - 1; ++t) o.w[NH / 2 + t] = f16_pack2(lo[2 * t], lo[2 * t + 1]);
    return o;
}
// The last word: 1 against the row's share of ||x||^2, and the half's part of c2 = ||c~||^2 against 1.
__device__ __forceinline__ uint32_t c2_word(float c2, int h, bool live) {
    const float hi = live ? (float)(_Float16)c2 : kPad8, lo = live ? c2 - hi : kPad8;
    return f16_pack2(1.0f, h == 0 ? hi : lo);
}

// Tables for k_assign_mfma8.  One workgroup per column block s, one thread per padded centroid
// (k <= 256).  Rows and centroids are scored relative to the mean of the block's centroids
// (distances do not change under a common shift, the rounding of the operands does).
// mfma8_prep_block is the work of one workgroup, given centroid j
// of the block in thread j's registers (zeros from k on); k_mfma8_prep reads the centroids from
// the codebook, the LBG loop's last update kernel has just computed them.
// COS: the centroids divided by their norms, about the origin (see cos_normalise).
template <bool COS = false>
__device__ __forceinline__ void mfma8_prep_block(float (&c)[8], int s, int j, int k, int nb,
                                                   u32x4 *__restrict__ atab, float *__restrict__ aux) {
    __shared__ float sh_red[3][4];
    __shared__ float sh_mu[4][8];
    float centre[8];
    float bad = 0.0f;
    bool zero = false;
    float *out = aux + (size_t)s * kMfma8Aux;
    float sg = kCosScale;
    if constexpr (COS) {
        bad = cos_normalise(c, zero);
#pragma unroll
        for (int t = 0; t < 8; ++t) {
            centre[t] = 0.0f;
            if (j == 0) out[t] = 0.0f;
        }
    } else {
        // centre: sum of c / 256 (no overflow for k <= 256), then * 256 / k
#pragma unroll
        for (int t = 0; t < 8; ++t) {
            float v = c[t] * 0.00390625f;
#pragma unroll
            for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off);
            if ((j & 63) == 0) sh_mu[j >> 6][t] = v;
        }
        __syncthreads();
        float p = 0.0f;
#pragma unroll
        for (int t = 0; t < 8; ++t) {
            centre[t] = (((sh_mu[0][t] + sh_mu[1][t]) + sh_mu[2][t]) + sh_mu[3][t]) * (256.0f / (float)k);
            if (j < k) c[t] -= centre[t];
            p = __builtin_fmaf(c[t] * 0.0625f, c[t] * 0.0625f, p);  // / 256
        }
#pragma unroll
        for (int off = 32; off > 0; off >>= 1) p += __shfl_xor(p, off);
        if ((j & 63) == 0) sh_red[2][j >> 6] = p;
        __syncthreads();
        sg = mfma8_scale((((sh_red[2][0] + sh_red[2][1]) + sh_red[2][2]) + sh_red[2][3]) * (256.0f / (float)k));
        if (j == 0) {
#pragma unroll
            for (int t = 0; t < 8; ++t) out[t] = -(centre[t] * sg);
        }
    }
    float mx = 0.0f, md = 0.0f;
    if (j < nb * 32) {
        const int b = j / 32, i = j % 32;
        u32x4 *dst = atab + ((size_t)s * nb + b) * 64;
        HalfOp<4> o[2];
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            float a[4];
#pragma unroll
            for (int t = 0; t < 4; ++t) a[t] = j < k ? -2.0f * (c[4 * h + t] * sg) : 0.0f;
            o[h] = half_op<4>(a);
        }
        // (a centroid of norm zero has the cosine distance 1: as far as any at a right angle)
        const float c2 = COS && zero ? kCosScale * kCosScale : o[0].n2 + o[1].n2;
        if (j < k) {
            mx = c2 + bad + (sg - sg);  // NaN: the block is not scored
            md = o[0].d2 + o[1].d2;
        }
#pragma unroll
        for (int h = 0; h < 2; ++h) dst[32 * h + i] = u32x4{o[h].w[0], o[h].w[1], o[h].w[2], c2_word(c2, h, j < k)};
    }
    // a NaN poisons the bound on purpose
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) {
        const float o = __shfl_xor(mx, off);
        mx = (mx == mx && o == o) ? fmaxf(mx, o) : __builtin_nanf("");
        md = fmaxf(md, __shfl_xor(md, off));
    }
    if ((j & 63) == 0) {
        sh_red[0][j >> 6] = mx;
        sh_red[1][j >> 6] = md;
    }
    __syncthreads();
    if (j == 0) {
        float r = sh_red[0][0], d = sh_red[1][0];
#pragma unroll
        for (int w = 1; w < 4; ++w) {
            const float o = sh_red[0][w];
            r = (r == r && o == o) ? fmaxf(r, o) : __builtin_nanf("");
            d = fmaxf(d, sh_red[1][w]);
        }
        out[8] = r;
        out[9] = d;
        out[10] = sg;
    }
}

template <bool COS = false>
static __global__ void __launch_bounds__(256) k_mfma8_prep(const float *__restrict__ cb, int m, int k, int nb,
                                                             u32x4 *__restrict__ atab, float *__restrict__ aux,
                                                             uint32_t *__restrict__ stat,
                                                             uint32_t *__restrict__ stat_next) {
    const int s = blockIdx.x, j = threadIdx.x;
    if (s == 0 && j < kStatSlots) stat[j * kStatStride] = stat_next[j * kStatStride] = 0u;
    float c[8];
#pragma unroll
    for (int t = 0; t < 8; ++t) c[t] = (j < k) ? cb[((size_t)s * k + j) * 8 + t] : 0.0f;
    mfma8_prep_block<COS>(c, s, j, k, nb, atab, aux);
}

// ---- the exact path of k_assign_mfma8 ---------------------------------------------------------
// Undecided rows of one (tile of 32 rows, column block) are decided by the whole wave in the
// reference's order (src/utils.rs:63-70, src/pq.rs:166-174): lane l owns centroids l, l + 64,
// l + 128, l + 192 (read from the wave's copy in LDS) and computes their distances to the row in
// sequential f32 order; the first of the smallest wins, as strict '<' over ascending indices gives.
// A NaN distance is never chosen unless it is centroid 0's, which is never replaced.  Euclidean
// compares the roots, as the reference does: the root is monotone, so the smallest root is that of the
// smallest square, and only a square within 2^-21 of it can share it; the others' roots are not taken.
// The row's floats come from the lanes that hold the tile (v_readlane): no memory access at all.  Read from
// memory again, eight rows to a round trip, and with every root taken: encode of 200,000 x 96 under cosine 93.5
// us, 88.0 so; of 300,000 x 128, k = 1024, 554 and 535; a fit of 1M x 128 with its encode 5.01 and 4.97 ms.
template <int CTRL> __device__ __forceinline__ uint32_t dpp_u32(uint32_t v) {
    return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, CTRL, 0xf, 0xf, false);
}
__device__ __forceinline__ uint32_t umin_u32(uint32_t a, uint32_t b) { return a < b ? a : b; }
// the smallest of all lanes' values, the same in every lane
__device__ __forceinline__ uint32_t wave_umin(uint32_t v) {
    v = umin_u32(v, dpp_u32<0xB1>(v));
    v = umin_u32(v, dpp_u32<0x4E>(v));
    v = umin_u32(v, dpp_u32<0x141>(v));
    v = umin_u32(v, dpp_u32<0x140>(v));
    uint32_t r = (uint32_t)__builtin_amdgcn_readlane((int)v, 0);
#pragma unroll
    for (int row = 1; row < 4; ++row) r = umin_u32(r, (uint32_t)__builtin_amdgcn_readlane((int)v, 16 * row));
    return r;
}

// A wave's copy of its block's centroids in LDS: two planes, one per half of a centroid, of 16 bytes per
// centroid.  The pick reads the four pieces of one run per lane, and the runs of the sixteen lanes of a read phase are
// to lie in different banks (with 32 bytes per centroid 38 % of the kernel's cycles were bank conflicts): 16 bytes
// stay free after every run, or, under cosine, where the norms need the room (40 KB per workgroup: four of
// them in a compute unit, cosine 86 -> 83 us), the order inside a run depends on the run.  Unused centroids are far off.
constexpr float kFar8 = 3e38f;
template <int METRIC> struct Lds8 {
    static constexpr bool SWZ = METRIC == M_COS;
    static constexpr int run_bytes = SWZ ? 64 : 80, plane = 64 * run_bytes;
    static __device__ __forceinline__ int run(int j, int h) {  // of the run's first centroid j
        return h * plane + (j >> 2) * run_bytes + (SWZ ? ((j >> 4) & 3) * 16 : 0);
    }
    static __device__ __forceinline__ float4 piece(const char *cl, int at, int i) {
        return *reinterpret_cast<const float4 *>(cl + (SWZ ? at ^ (i * 16) : at + i * 16));
    }
    static __device__ __forceinline__ float4 half(const char *cl, int j, int h) { return piece(cl, run(j & ~3, h), j & 3); }
    static __device__ __forceinline__ void set(char *cl, int j, int h, float4 v) {
        const int at = run(j & ~3, h), i = j & 3;
        *reinterpret_cast<float4 *>(cl + (SWZ ? at ^ (i * 16) : at + i * 16)) = v;
    }
    static __device__ __forceinline__ void load(const char *cl, int j, float (&c)[8]) {
        const float4 a = half(cl, j, 0), b = half(cl, j, 1);
        c[0] = a.x, c[1] = a.y, c[2] = a.z, c[3] = a.w, c[4] = b.x, c[5] = b.y, c[6] = b.z, c[7] = b.w;
    }
};

// cl: the column block's centroids in LDS (this wave's copy).
// todo: ballot of the lanes (below 32) whose row is undecided; xr: the lane's row.
// Returns the codes of those rows in their lanes, and their distances in dist (other lanes keep
// `code` and `dist`).
template <int METRIC>
__device__ __forceinline__ int exact_rows8(unsigned long long todo, int code, float &dist, const char *cl,
                                           const float *norms, const float (&xr)[8], int k, int lane) {
    constexpr uint32_t kInfKey = METRIC == M_COS ? 0xff800000u : 0x7f800000u;  // sort key of +inf
    while (todo) {
        const int src = __builtin_amdgcn_readfirstlane(__ffsll(todo) - 1);
        todo &= todo - 1;
        float xs[8];
#pragma unroll
        for (int d = 0; d < 8; ++d) xs[d] = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(xr[d]), src));
        const float na = METRIC == M_COS ? seq_norm8(xs) : 0.0f;
        // sort keys of the lane's four distances (Euclidean: of the squares); a NaN sorts behind +inf
        uint32_t key[4];
        float first = 0.0f;
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const int j = lane + 64 * q;
            float c[8];
            Lds8<METRIC>::load(cl, j, c);
            const float d = dist8<METRIC == M_COS ? M_COS : M_SQ>(xs, c, na, METRIC == M_COS ? norms[j] : 0.0f);
            if (q == 0) first = d;
            key[q] = j < k && d == d ? dist_key<METRIC>(d) : 0xffffffffu;
        }
        const uint32_t best_key = wave_umin(umin_u32(umin_u32(key[0], key[1]), umin_u32(key[2], key[3])));
        const float d0 = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(first), 0));
        int best = 0;
        float bd = METRIC == M_EUCLID ? sqrtf(d0) : d0;  // centroid 0 where nothing is below +inf
        if (d0 == d0 && best_key < kInfKey) {  // uniform
            unsigned long long at[4];
            bd = key_dist<METRIC>(best_key);
            if constexpr (METRIC == M_EUCLID) {
                const uint32_t close = __float_as_uint(__builtin_fmaf(bd, 4.76837158203125e-07f, bd));
                bd = sqrtf(bd);
#pragma unroll
                for (int q = 0; q < 4; ++q) at[q] = __ballot(key[q] <= close);
                if (__popcll(at[0]) + __popcll(at[1]) + __popcll(at[2]) + __popcll(at[3]) > 1) {
#pragma unroll
                    for (int q = 0; q < 4; ++q) at[q] = __ballot(key[q] <= close && sqrtf(__uint_as_float(key[q])) == bd);
                }
            } else {
#pragma unroll
                for (int q = 0; q < 4; ++q) at[q] = __ballot(key[q] == best_key);
            }
            best = at[0] ? __ffsll(at[0]) - 1 : at[1] ? __ffsll(at[1]) + 63 : at[2] ? __ffsll(at[2]) + 127 : __ffsll(at[3]) + 191;
        }
        if (lane == src) {
            code = best;
            dist = bd;  // the chosen centroid's distance as computed
        }
    }
    return code;
}

// The tables of mfma8_prep_block made by one wave for itself (the same operands up to the order in
// which the sums for the centre and the scale are added, which any centre and scale allow): lane (r, h) makes its
// own operands of the centroids 32 b + r, dimensions [4h, 4h + 4), from the wave's copy of the centroids in LDS.
// COS: of the centroids divided by their norms (norms: one per centroid, in LDS).
template <bool COS>
__device__ __forceinline__ void own_operands(const char *cl, const float *norms, int k, int nb, int r, int h,
                                             u32x4 (&A)[8], float (&muh)[4], float &mc2, float &mdc, float &sg) {
    float cv[8][4];
    float sum[4] = {0.f, 0.f, 0.f, 0.f};
    float bad = 0.0f;
    sg = kCosScale;
#pragma unroll
    for (int b = 0; b < 8; ++b) {
        const int j = 32 * b + r;
        const float4 v = Lds8<COS ? M_COS : M_SQ>::half(cl, j, h);
        cv[b][0] = v.x, cv[b][1] = v.y, cv[b][2] = v.z, cv[b][3] = v.w;
#pragma unroll
        for (int u = 0; u < 4; ++u) sum[u] += j < k ? cv[b][u] * 0.00390625f : 0.0f;  // no overflow for k <= 256
    }
    if constexpr (!COS) {
#pragma unroll
        for (int u = 0; u < 4; ++u) {
#pragma unroll
            for (int off = 16; off > 0; off >>= 1) sum[u] += __shfl_xor(sum[u], off);  // over the lanes of this half
            sum[u] *= 256.0f / (float)k;  // the centre
        }
        float p = 0.0f;
#pragma unroll
        for (int b = 0; b < 8; ++b)
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                const float c = 32 * b + r < k ? (cv[b][u] - sum[u]) * 0.0625f : 0.0f;
                p = __builtin_fmaf(c, c, p);
            }
#pragma unroll
        for (int off = 32; off > 0; off >>= 1) p += __shfl_xor(p, off);
        sg = mfma8_scale(p * (256.0f / (float)k));
        bad = sg - sg;  // 0 or NaN
    }
#pragma unroll
    for (int u = 0; u < 4; ++u) muh[u] = COS ? 0.0f : -(sum[u] * sg);
    float mx = 0.0f, md = 0.0f;
#pragma unroll
    for (int b = 0; b < 8; ++b) {
        if (b >= nb) {  // uniform; never multiplied
            A[b] = A[0];
            continue;
        }
        const bool live = 32 * b + r < k;
        float scale = -2.0f * sg, c2, d2;
        const float nc = COS && live ? norms[32 * b + r] : 0.0f;
        if constexpr (COS) {
            scale = nc == 0.0f ? 0.0f : -2.0f * (1.0f / nc);
            bad = nc == 0.0f || (nc >= 1e-15f && nc <= 1e15f) ? 0.0f : __builtin_nanf("");
        }
        float a[4];
#pragma unroll
        for (int u = 0; u < 4; ++u)
            a[u] = !live ? 0.0f : COS ? (scale * cv[b][u]) * kCosScale : scale * (cv[b][u] - sum[u]);
        const HalfOp<4> o = half_op<4>(a);
        int pa, pb;
        swap_halves(__float_as_int(o.n2), pa, pb);
        c2 = COS && nc == 0.0f ? kCosScale * kCosScale : __int_as_float(pa) + __int_as_float(pb);
        swap_halves(__float_as_int(o.d2), pa, pb);
        d2 = __int_as_float(pa) + __int_as_float(pb);
        const float cx = live ? c2 + bad : 0.0f;
        mx = (mx == mx && cx == cx) ? fmaxf(mx, cx) : __builtin_nanf("");
        md = fmaxf(md, live ? d2 : 0.0f);
        A[b] = u32x4{o.w[0], o.w[1], o.w[2], c2_word(c2, h, live)};
    }
#pragma unroll
    for (int off = 16; off > 0; off >>= 1) {
        const float o = __shfl_xor(mx, off);
        mx = (mx == mx && o == o) ? fmaxf(mx, o) : __builtin_nanf("");
        md = fmaxf(md, __shfl_xor(md, off));
    }
    mc2 = mx;
    mdc = md;
}

// The row operand of a tile: the lane's NH dimensions relative to the centre (cosine: of length kCosScale), as
// HalfOp's slots want them.
template <int NH> struct RowOp {
    u32x4 b16[NH / 4];
    float e2;                    // what the rounding lost, squared, both halves
    float x2 = 0.0f, rx = 0.0f;  // cosine: ||x||^2 and 1 / ||x|| of the row as it is
};
template <int METRIC, int NH>
__device__ __forceinline__ RowOp<NH> row_op(const float (&xraw)[NH], float sg, const float (&muh)[NH]) {
    RowOp<NH> o;
    float xv[NH];
    int pa, pb;
    float p = 0.0f, d2 = 0.0f;
    if constexpr (METRIC == M_COS) {
#pragma unroll
        for (int u = 0; u < NH; ++u) p = __builtin_fmaf(xraw[u], xraw[u], p);
        swap_halves(__float_as_int(p), pa, pb);
        o.x2 = __int_as_float(pa) + __int_as_float(pb);
        o.rx = __builtin_amdgcn_rsqf(o.x2);
        const float f = kCosScale * o.rx;
#pragma unroll
        for (int u = 0; u < NH; ++u) xv[u] = xraw[u] * f;
        p = 0.0f;
    } else {
#pragma unroll
        for (int u = 0; u < NH; ++u) xv[u] = __builtin_fmaf(xraw[u], sg, muh[u]);
    }
#pragma unroll
    for (int u = 0; u < NH; ++u) p = __builtin_fmaf(xv[u], xv[u], p);
    using h2 = _Float16 __attribute__((ext_vector_type(2)));
    uint32_t w[NH];
#pragma unroll
    for (int u = 0; u < NH / 2; ++u) {
        w[u] = __builtin_bit_cast(uint32_t, __builtin_convertvector((floatx2{xv[2 * u], xv[2 * u + 1]}), h2));
        float dl, dh;  // x~ - x: one instruction each that reads a half of the pair
        asm("v_fma_mix_f32 %0, %1, 1.0, -%2 op_sel_hi:[1,0,0]" : "=v"(dl) : "v"(w[u]), "v"(xv[2 * u]));
        asm("v_fma_mix_f32 %0, %1, 1.0, -%2 op_sel:[1,0,0] op_sel_hi:[1,0,0]" : "=v"(dh) : "v"(w[u]), "v"(xv[2 * u + 1]));
        d2 = __builtin_fmaf(dl, dl, d2);
        d2 = __builtin_fmaf(dh, dh, d2);
    }
    swap_halves(__float_as_int(d2), pa, pb);
    o.e2 = __int_as_float(pa) + __int_as_float(pb);
#pragma unroll
    for (int u = 0; u < NH / 2 - 1; ++u) w[NH / 2 + u] = w[u];
    w[NH - 1] = __builtin_bit_cast(uint32_t, __builtin_convertvector((floatx2{p * kLift8, 1.0f}), h2));
#pragma unroll
    for (int i = 0; i < NH / 4; ++i) o.b16[i] = u32x4{w[4 * i], w[4 * i + 1], w[4 * i + 2], w[4 * i + 3]};
    return o;
}
// Whether the best of the two smallest keys has won (false for NaN / inf - inf); e2c: the centroids' share of
// the rounding, acc8: 3 * NH / 4 * 2^-16 max ||c~||^2 (||x||^2 <= 2 (s2 + ||c||^2) stands for the row's norm).
template <int METRIC, int NH>
__device__ __forceinline__ bool decided8(float s1, float s2, const RowOp<NH> &row, float e2c, float acc8) {
    const float E = (row.e2 + kFlush8 * (NH / 4)) + e2c;
    const float margin = __builtin_fmaf(4.001f, __builtin_amdgcn_sqrtf(2.0f * s2 * E), __builtin_fmaf(8.0f, E, acc8)) +
                         (6.103515625e-05f + NH / 4 * 3.0517578125e-05f) * s2;
    // 1.2e5: below every padding centroid
    return (s2 - s1) > margin && s1 < 1.2e5f && (METRIC != M_COS || (row.x2 > 1e-30f && row.x2 < 1e30f));
}
// A lane half's share of the distance to a centroid: NH dimensions, fused.  Cosine: of the inner product.
template <int METRIC, int NH> __device__ __forceinline__ float share8(const float (&xraw)[NH], const float (&c)[NH]) {
    if constexpr (METRIC == M_COS) {
        float p = xraw[0] * c[0];
#pragma unroll
        for (int u = 1; u < NH; ++u) p = __builtin_fmaf(xraw[u], c[u], p);
        return p;
    } else {
        float d = xraw[0] - c[0], p = d * d;
#pragma unroll
        for (int u = 1; u < NH; ++u) {
            d = xraw[u] - c[u];
            p = __builtin_fmaf(d, d, p);
        }
        return p;
    }
}

// One wave = one column block of 8 floats against a run of tiles of 32 rows.  The wave keeps the
// A operands of all the block's centroids in registers (8 blocks of 32 centroids x 4 registers) and a copy of the block's centroids in LDS, and streams the rows past them: the
// inner loop reads no memory.  A lane's 16 scores of a tile are four runs of four consecutive
// centroids; the smallest score of a run, tagged with the run's first index, is the run's key, and
// the smallest and second-smallest key of the row are kept (two minima and one v_and_or per run,
// five v_min3 / v_med3 per four runs: 17 vector instructions for 16 scores).  When the two best
// keys are further apart than the error bound, every centroid outside the best run is provably
// further from the row than the run's best one, and the reference's choice is the first smallest
// exact distance among the run's four centroids.  Each lane half sums its four dimensions of all four with fused
// multiply-adds; the smallest sum decides where it is clear of the second, else the run is gone through
// in the reference's order.  (Two full chains of rounded products per half, and two roots under Euclidean,
// took 46 to 75 vector instructions where this takes 36: a pass of a fit over 1M x 16 blocks 340 -> 320 us, fit and
// encode of 1M x 128 4.61 -> 4.42 ms.)  Otherwise the row goes through the reference-order argmin.
// Bound by vector-instruction issue: 275 per tile and column block, half of them the selection's, 2.1 GHz.
// SG = 4: the four waves of a workgroup take the four column blocks of one 128-byte line of the
// same rows.  SG = 1 (m not a multiple of 4): the four waves take consecutive runs of one block.
// FULL: 8 blocks of 32 centroids (k above 224), scored without a branch between them.
// OWN: every wave makes the operands, the centre and the bound of its block from the centroids it
// holds in LDS, about 700 vector instructions, instead of reading the tables that k_mfma8_prep has
// made: for grids of one round of workgroups, where that launch (6.5 us) is in the way.
template <int METRIC, bool LBG, int SG, bool FULL, bool OWN = false>
__global__ void __launch_bounds__(256, 3) k_assign_mfma8(AssignArgs a, Mfma8Tables tb, int run_tiles, int64_t nruns,
                                                            int64_t run_stride) {
    constexpr int SD = 8;
    __shared__ __attribute__((aligned(16))) char lds_cb[4][2 * Lds8<METRIC>::plane];
    __shared__ float lds_norm[METRIC == M_COS ? 4 : 1][METRIC == M_COS ? 512 : 1];  // the centroids' norms, then their reciprocals
    // the wave's number through readfirstlane: what follows from it (column block, first row, base
    // addresses) is then uniform for the compiler and lives in scalar registers
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const int r = lane & 31, h = lane >> 5;
    const int nb = FULL ? 8 : tb.nb, m = a.m, k = a.k;
    // Workgroups are dealt round-robin to the 8 XCDs, each with its own L2: workgroups id, id + 8,
    // id + 16, ... (the same XCD, dispatched close together) take the column-block groups of one
    // run of rows, so that the code bytes of a row are merged in one L2 before they are written back.
    const int ngroups = m / SG;
    const unsigned per_chunk = 8u * (unsigned)ngroups;
    const unsigned chunk_id = blockIdx.x / per_chunk, rem = blockIdx.x % per_chunk;
    const int g = (int)(rem / 8u);
    const int64_t run_first = (int64_t)chunk_id * 8 + (rem % 8u);
    const int s = SG == 4 ? g * 4 + wave : g;
    if (run_first >= nruns) return;
    if constexpr (LBG) {
        if (__builtin_amdgcn_readfirstlane((int)block_done(a, s))) return;  // the block has converged
    }

    // the block's centroids: this wave's copy in LDS (no other wave reads it: no barrier)
    char *cl = lds_cb[wave];
    {
        const float4 *src = reinterpret_cast<const float4 *>(a.cb + (size_t)s * k * SD);
        const int nv = 2 * k;
#pragma unroll
        for (int c = 0; c < 8; ++c) {
            const int i = lane + 64 * c;
            const float4 v = src[i < nv ? i : 0];
            Lds8<METRIC>::set(cl, i >> 1, i & 1, i < nv ? v : make_float4(kFar8, kFar8, kFar8, kFar8));
        }
    }
    float *norms = lds_norm[METRIC == M_COS ? wave : 0];
    if constexpr (METRIC == M_COS) {
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const int j = lane + 64 * q;
            float c[8];
            Lds8<METRIC>::load(cl, j, c);
            norms[j] = seq_norm8(c);
            norms[256 + j] = norms[j] == 0.0f ? 0.0f : 1.0f / norms[j];
        }
    }
    // the A operands of every block of 32 centroids, the centre's dimensions [4h, 4h + 4), the bound
    u32x4 A[8];
    float muh[4];
    float mc2, mdc, sg;
    if constexpr (OWN) {
        if (blockIdx.x == 0)
            for (int i = threadIdx.x; i < kStatSlots; i += 256) tb.stat_next[i * kStatStride] = 0u;
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        own_operands<METRIC == M_COS>(cl, norms, k, nb, r, h, A, muh, mc2, mdc, sg);
    } else {
        const u32x4 *ap = tb.atab + (size_t)s * nb * 64 + lane;
#pragma unroll
        for (int b = 0; b < 8; ++b) A[b] = ap[(size_t)(b < nb ? b : 0) * 64];
        const float *aux = tb.aux + (size_t)s * kMfma8Aux;
#pragma unroll
        for (int u = 0; u < 4; ++u) muh[u] = aux[4 * h + u];
        mc2 = aux[8];
        mdc = aux[9];
        sg = aux[10];
    }
    const uint32_t keep = opaque_vgpr(0xFFFFFF00u);
    const float acc8 = 4.57763671875e-05f * mc2;  // 2^-16 * 3: see the margin
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();

    uint32_t n_exact = 0;
    bool chg = false;
    // The workgroup walks over its runs of rows (run_first, run_first + run_stride, ...) with the
    // operands it has loaded: the grid is a few workgroups per compute unit, not one per run.
    for (int64_t run_id = run_first; run_id < nruns; run_id += run_stride) {
    const int64_t tile0 = SG == 4 ? run_id * run_tiles : (run_id * 4 + wave) * run_tiles;
    const int64_t row0 = tile0 * 32;
    if (row0 >= a.n) break;  // SG == 1: the last run may end before this wave's share
    const int64_t left = (a.n - row0 + 31) / 32;
    const int ntiles = (int)(left < run_tiles ? left : run_tiles);
    // rows two tiles ahead.  Addresses are a scalar base (the run's first row) plus a 32-bit lane
    // offset that moves on by 32 rows per tile (the host keeps the run's extent below 2^31 bytes).
    const float *xrun = a.x + row0 * a.ld + (int64_t)s * SD;          // uniform
    const uint8_t *crun = a.codes + (size_t)s * a.n + row0;           // uniform (LBG: [m][n] codes)
    const int64_t lane_rows = a.n - (row0 + r);                       // rows from this lane's first to the end
    const int64_t lane_left = lane_rows > 0 ? (lane_rows + 31) / 32 : 0;
    // tiles of this run in which the lane has a row; the fetches past the run's end read the run's
    // first row (the next run belongs to a workgroup on another XCD: its rows would be fetched into two L2s)
    const int lane_tiles = (int)(lane_left < run_tiles ? lane_left : run_tiles);
    const uint32_t xstep = 128u * (uint32_t)a.ld;                                          // bytes per tile
    uint32_t xoff = 4u * ((uint32_t)r * (uint32_t)a.ld + 4u * (uint32_t)h), coff = (uint32_t)r;  // of the lane's row in tile 0
    // rows may start at any float (any leading dimension): a 16-byte load that only claims 4-byte alignment
    typedef float rowpiece __attribute__((ext_vector_type(4), aligned(4)));
    auto fetch_x = [&](int t) {
        const char *p = reinterpret_cast<const char *>(xrun) + (t < lane_tiles ? xoff : 16u * (uint32_t)h);
        const rowpiece v = *reinterpret_cast<const rowpiece *>(p);
        return make_float4(v[0], v[1], v[2], v[3]);
    };
    auto fetch_c = [&](int t) { return crun[t < lane_tiles ? coff : 0u]; };
    float4 xa = fetch_x(0);
    uint8_t oa = 0, ob = 0;
    if constexpr (LBG) oa = fetch_c(0);
    xoff += xstep;
    coff += 32;
    float4 xb = fetch_x(1);
    if constexpr (LBG) ob = fetch_c(1);
    for (int t = 0; t < ntiles; ++t) {
        const float4 xc = xa;
        const uint8_t old = oa;
        xa = xb;
        oa = ob;
        xoff += xstep;
        coff += 32;
        xb = fetch_x(t + 2);
        if constexpr (LBG) ob = fetch_c(t + 2);
        const float xraw[4] = {xc.x, xc.y, xc.z, xc.w};
        const RowOp<4> row = row_op<METRIC, 4>(xraw, sg, muh);
        const u32x4 xb16 = row.b16[0];
        int m1 = 0x7f800000, m2 = 0x7f800000;  // +inf
        // One block of 32 centroids.  The tag leaves out the lane half (bit 2), so it is the same in
        // every lane and lives in scalar registers.
        // The scores of block b + 1 are made while block b's go through the selection: a matrix
        // instruction holds back the vector instructions of OTHER waves of its SIMD for as long as it
        // runs, but independent vector instructions of its own wave issue in its shadow, so every
        // matrix instruction is followed by a block's selection from the same wave.
#define VQ_MFMA(b, acc)                                                                                         \
    acc = __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(f16x8, A[b]), __builtin_bit_cast(f16x8, xb16), \
                                                 zero, 0, 0, 0);
#define VQ_RUN_KEY(b, acc, p)                                                                                   \
    {                                                                                                           \
        const int gmin = imin(imin(imin(__float_as_int(acc[4 * p]), __float_as_int(acc[4 * p + 1])),            \
                                   __float_as_int(acc[4 * p + 2])),                                             \
                              __float_as_int(acc[4 * p + 3]));                                                  \
        key[p] = (int)(((uint32_t)gmin & keep) | (uint32_t)(32 * (b) + 8 * p));                                 \
    }
        // selection of block b (scores in cur) with the matrix instructions of block nb (into nxt) in between
#define VQ_SCORE_BLOCK(b, cur, nb, nxt, more)                                                                   \
    {                                                                                                           \
        int key[4];                                                                                             \
        if (more) { VQ_MFMA(nb, nxt) }                                                                          \
        __builtin_amdgcn_sched_barrier(0);                                                                      \
        VQ_RUN_KEY(b, cur, 0) VQ_RUN_KEY(b, cur, 1) VQ_RUN_KEY(b, cur, 2) VQ_RUN_KEY(b, cur, 3)                  \
        top2_push4(m1, m2, key[0], key[1], key[2], key[3]);                                                     \
        __builtin_amdgcn_sched_barrier(0);                                                                      \
    }
        const floatx16 zero = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
        floatx16 accA, accB;
        VQ_MFMA(0, accA)
        if constexpr (FULL) {
            VQ_SCORE_BLOCK(0, accA, 1, accB, true) VQ_SCORE_BLOCK(1, accB, 2, accA, true)
            VQ_SCORE_BLOCK(2, accA, 3, accB, true) VQ_SCORE_BLOCK(3, accB, 4, accA, true)
            VQ_SCORE_BLOCK(4, accA, 5, accB, true) VQ_SCORE_BLOCK(5, accB, 6, accA, true)
            VQ_SCORE_BLOCK(6, accA, 7, accB, true) VQ_SCORE_BLOCK(7, accB, 0, accA, false)
        } else {
            VQ_SCORE_BLOCK(0, accA, 1, accB, true)
            if (nb > 2) {
                VQ_SCORE_BLOCK(1, accB, 2, accA, true) VQ_SCORE_BLOCK(2, accA, 3, accB, true)
                if (nb > 4) {
                    VQ_SCORE_BLOCK(3, accB, 4, accA, true) VQ_SCORE_BLOCK(4, accA, 5, accB, true)
                    if (nb > 6) {
                        VQ_SCORE_BLOCK(5, accB, 6, accA, true) VQ_SCORE_BLOCK(6, accA, 7, accB, true)
                        VQ_SCORE_BLOCK(7, accB, 0, accA, false)
                    } else {
                        VQ_SCORE_BLOCK(5, accB, 0, accA, false)
                    }
                } else {
                    VQ_SCORE_BLOCK(3, accB, 0, accA, false)
                }
            } else {
                VQ_SCORE_BLOCK(1, accB, 0, accA, false)
            }
        }
#undef VQ_MFMA
#undef VQ_RUN_KEY
#undef VQ_SCORE_BLOCK
        // the partner lane (other half) saw the other 16 centroids of every block
        m1 |= 4 * h;  // bit 2 of the centroid index: the lane half
        m2 |= 4 * h;
        int f1, g1, f2, g2;
        swap_halves(m1, f1, g1);
        swap_halves(m2, f2, g2);
        const float s1 = __int_as_float(imin(f1, g1));
        const float s2 = __int_as_float(imin(imax(f1, g1), imin(f2, g2)));
        const bool mine = h == 0 && t < lane_tiles;  // the lane's row of this tile exists
        const bool near = decided8<METRIC, 4>(s1, s2, row, mdc, acc8);
        const int first = (int)(__float_as_uint(s1) & 0xFCu);  // first centroid of the best run
        // The best of the run's four centroids.  Each lane half takes its four dimensions of all of them (fused
        // multiply-adds), the halves' sums meet two centroids each; the smallest that is clear of the second by
        // 2^-17, more than this sum and the reference's round, is the reference's choice.
        int code;
        bool clear;
        {
            const int run = Lds8<METRIC>::run(first, h);
            float p[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const float4 v = Lds8<METRIC>::piece(cl, run, i);
                p[i] = share8<METRIC, 4>(xraw, {v.x, v.y, v.z, v.w});
            }
            // lower half: centroids first, first + 1; upper half: first + 2, first + 3
            const auto r02 = __builtin_amdgcn_permlane32_swap(__float_as_int(p[0]), __float_as_int(p[2]), false, false);
            const auto r13 = __builtin_amdgcn_permlane32_swap(__float_as_int(p[1]), __float_as_int(p[3]), false, false);
            float da = __int_as_float((int)r02[0]) + __int_as_float((int)r02[1]);
            float db = __int_as_float((int)r13[0]) + __int_as_float((int)r13[1]);
            const int j0 = first + 2 * h;
            int ka, kb;  // sort keys: non-negative distances as they are
            if constexpr (METRIC == M_COS) {
                // 1 - cos (a centroid of norm zero: 1), lifted so that rounding leaves it positive
                const float2 inv = *reinterpret_cast<const float2 *>(norms + 256 + j0);
                da = __builtin_fmaf(-(da * row.rx), inv.x, 1.001f);
                db = __builtin_fmaf(-(db * row.rx), inv.y, 1.001f);
                ka = j0 < k ? __float_as_int(da) : 0x7f800000;
                kb = j0 + 1 < k ? __float_as_int(db) : 0x7f800000;
            } else {
                ka = __float_as_int(da);
                kb = __float_as_int(db);
            }
            int lo = imin(ka, kb), hi = imax(ka, kb), at = j0 + (kb < ka ? 1 : 0);
            int l0, l1, h0, h1, a0, a1;
            swap_halves(lo, l0, l1);
            swap_halves(hi, h0, h1);
            swap_halves(at, a0, a1);
            code = l1 < l0 ? a1 : a0;  // (lower half: 0 its own, 1 the partner's)
            const float best = __int_as_float(imin(l0, l1));
            const float second = __int_as_float(imin3(imax(l0, l1), h0, h1));
            // (1e-36: sums of squares in the subnormal range)
            if constexpr (METRIC == M_COS)
                clear = second - best > 7.62939453125e-06f;
            else
                clear = __builtin_fmaf(second, 0.99999237060546875f, -1e-36f) > best;
        }
        const unsigned long long todo = __ballot(mine && !near), ties = __ballot(mine && near && !clear);
        float dist = 0.0f;  // of the chosen centroid, as the reference computes it (where it is asked for)
        bool want_dist = false;
        if constexpr (!LBG) want_dist = a.dist != nullptr;
        if ((todo | ties) != 0 || want_dist) {  // the same in every lane
            float xs[8];  // the lane's row
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                int lo, hi;
                swap_halves(__float_as_int(xraw[u]), lo, hi);
                xs[u] = __int_as_float(lo);
                xs[4 + u] = __int_as_float(hi);
            }
            const float na = METRIC == M_COS ? seq_norm8(xs) : 0.0f;
            if (ties) {
                // the run's four centroids in the reference's order: the first of the smallest
                float bd = 0.0f;
                int bj = first;
                for (int i = 0; i < 4; ++i) {
                    float c[8];
                    Lds8<METRIC>::load(cl, first + i, c);
                    const float d = dist8<METRIC>(xs, c, na, METRIC == M_COS ? norms[first + i] : 0.0f);
                    if (i == 0 || (first + i < k && d < bd)) {
                        bd = d;
                        bj = first + i;
                    }
                }
                code = clear ? code : bj;
            }
            if (want_dist) {
                float c[8];
                Lds8<METRIC>::load(cl, code, c);
                dist = dist8<METRIC>(xs, c, na, METRIC == M_COS ? norms[code] : 0.0f);
            }
            if (todo) {  // the reference-order argmin of the undecided rows
                n_exact += (uint32_t)__popcll(todo);
                code = exact_rows8<METRIC>(todo, code, dist, cl, norms, xs, k, lane);
            }
        }
        if (mine) {
            const uint32_t rr = 32u * (uint32_t)t + (uint32_t)r;  // row within the run
            if constexpr (LBG) {
                if (old != (uint8_t)code) {
                    a.codes[(size_t)s * a.n + row0 + rr] = (uint8_t)code;
                    chg = true;
                }
            } else {
                const size_t out0 = (size_t)row0 * m + s;  // uniform
                a.codes[out0 + rr * (uint32_t)m] = (uint8_t)code;
                if (a.dist) a.dist[out0 + rr * (uint32_t)m] = dist;  // for the caller that merges chunks of a larger codebook
                if (a.out16) {  // the reconstruction, round to nearest even
                    const float4 c0 = Lds8<METRIC>::half(cl, code, 0), c1 = Lds8<METRIC>::half(cl, code, 1);
                    auto two = [](float lo, float hi) {
                        return (uint32_t)__half_as_ushort(__float2half_rn(lo)) | ((uint32_t)__half_as_ushort(__float2half_rn(hi)) << 16);
                    };
                    reinterpret_cast<u32x4 *>(a.out16)[out0 + rr * (uint32_t)m] =
                        u32x4{two(c0.x, c0.y), two(c0.z, c0.w), two(c1.x, c1.y), two(c1.z, c1.w)};
                }
            }
        }
    }
    }  // runs
    if constexpr (LBG) {
        // changed[s]: one lane per wave, once per wave, and only where the flag still reads 0 (every
        // store to one address is serialised in its L2 channel; a stale 0 from the vector cache
        // costs a store, nothing else).
        if (__any(chg) && lane == 0 && a.changed[s] == 0) a.changed[s] = 1;
    }
    if (lane == 0 && n_exact)
        atomicAdd(tb.stat + ((run_first * 4 + wave) & (kStatSlots - 1)) * kStatStride, n_exact);
}

}  // namespace vq

// ---- column blocks of any other width, on the kernels for multiples of 8 -------------------------
namespace vq {

// y[i][s][t] = x[i][s * sd + t] for t < sd, zeros up to sdp (a multiple of 8).  Rows and centroids
// padded alike keep every distance bit for bit — the padding adds (0 - 0)^2 = +0.0 to sums that are
// never -0.0 — so a block of 10 components runs on the kernels for 16.  One thread makes one
// 16-byte piece, four pieces per thread; a workgroup's 1024 pieces are consecutive, so the reads of
// a wave cover whole lines of the rows although a piece's floats may start anywhere.  Bound by HBM.
// Training of 60,007 x 100 in blocks of 10, k = 200, ten iterations and the encode: 45.2 -> 1.69 ms.
static __global__ void __launch_bounds__(256) k_pad_blocks(const float *__restrict__ x, int64_t n, int64_t ld, int m,
                                                           int sd, int sdp, float *__restrict__ y) {
    const uint32_t per_block = (uint32_t)sdp / 4u, per_row = per_block * (uint32_t)m;
    const int64_t first = (int64_t)blockIdx.x * 1024;
    const int64_t row0 = first / per_row;  // uniform
    const uint32_t rem0 = (uint32_t)(first - row0 * per_row);
    float v[4][4];
    int64_t row[4];
#pragma unroll
    for (int u = 0; u < 4; ++u) {
        const uint32_t local = rem0 + threadIdx.x + 256u * u;
        const uint32_t dr = local / per_row, c = local - dr * per_row;
        const uint32_t s = c / per_block, t = 4u * (c - s * per_block);
        row[u] = row0 + dr;
        const float *p = x + (row[u] < n ? row[u] : n - 1) * ld + (int64_t)s * sd;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const float w = p[t + e < (uint32_t)sd ? t + e : 0u];
            v[u][e] = t + e < (uint32_t)sd ? w : 0.0f;
        }
    }
#pragma unroll
    for (int u = 0; u < 4; ++u)
        if (row[u] < n) reinterpret_cast<float4 *>(y)[first + threadIdx.x + 256 * u] = make_float4(v[u][0], v[u][1], v[u][2], v[u][3]);
}

// The other direction for the codebooks: out[i][t] = y[i][t], t < sd.
static __global__ void __launch_bounds__(256) k_unpad_rows(const float *__restrict__ y, int64_t n, int sd, int sdp,
                                                           float *__restrict__ out) {
    const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    if (i < n * sd) out[i] = y[i / sd * sdp + i % sd];
}

}  // namespace vq

// =============================================================================================
// Wide column blocks (sub_dim a multiple of 8, up to the full dimension: RVQ stages).
namespace vq {

// ---------------------------------------------------------------------------------------------
// Wide column blocks on the bf16 matrix cores: the operand split of k_assign_mfma8 applied to
// 16 dimensions at a time.  With the high and low bf16 parts of the centroid operand (ah, al) and
// of the row operand (xh, xl), a tile of 32 rows x 32 centroids takes three instructions per 16
// dimensions, ah.xh + al.xh + ah.xl, each with all 16 contraction slots in use (each lane half
// owns 8 of the 16 dimensions).  An earlier shape worked on 8 dimensions with two instructions,
// {ah, al}.{xh, xh} and {ah, al}.{xl, 0}: a quarter of the slots multiplied zeros.
// A workgroup = 128 rows; a wave takes one tile of 32 rows against every tile of 32 centroids: 8
// accumulator tiles (128 registers) that start at ||c - mu||^2.  The centroid operands of a tile
// are the 16 bytes of ah and the 16 bytes of al as they lie in LDS, and the row is split once per
// 16 dimensions for 3 NB matrix instructions, so no operand is assembled in registers (vector
// and matrix instructions take turns on a SIMD).  ||x - mu||^2 is summed on the vector ALU and
// added to the scores before the selection.  The A operands of 16 dimensions (16 KB for 256
// centroids) are staged in LDS once per workgroup, double-buffered; the next A operands are
// fetched one stage ahead, the row two.
// What decides (x and c relative to the centre, t = kWideT): a score is off by no more than
//   A ||c||^2 + (S + A) 2 ||x|| ||c||,  S = 3 * 2^-16 (split, as above),  A = (27 sd/8 + 28) * 2^-24
// (fp32 accumulation, an upper bound: at most 17 additions per instruction, 1.5 instructions per 8
// dimensions, the sum of ||c||^2, the rounding of x - mu and c - mu), and 2 ||x|| ||c|| <= t ||x||^2 +
// ||c||^2 / t.  The share of the row is the same for every centroid; the share of the centroid, pen[j],
// is taken off its score before the selection.  A centroid whose lowered score is clear of the best one
// by both rows' shares, 2 pen[best], the tag (2^-14 of the score) and the reference's own rounding
// (2 (sd + 16) * 2^-24 of the distance) has lost.  A bound from the LARGEST ||c|| of the block listed 7-20 %
// of the rows of a late residual stage (up to 7 % of them for all centroids, 0.65 ms per pass at
// 1M x 256, 194 us on average, now 15-25; the fit of 8 stages 80 -> 65 ms): there most rows choose between a few centroids of small norm beside many of large norm.
// t is a compromise: the undecided share is flat between 0.25 and 0.7 (it doubles outside).
constexpr float kWideT = 0.35f;

// HALF: one product of binary16 operands instead of three of bf16 parts.  Rows and centroids are scaled by
// a power of two that brings the centroids' root mean square norm to 32 ... 64; what the rounding of a row
// (dx = ||x - xh||, summed as it happens) and of a centroid (dc) can do is 2 dx ||c|| + 2 ||x|| dc, split
// between the row and the centroid as above, with kWideRho the usual dx / ||x||:
//   (x c - xh ch = (x - xh) ch + x (c - ch));  2 dx ||c|| <= dx^2 t / rho + ||c||^2 rho / t,   2 ||x|| dc <= ||x||^2 rho t + dc^2 / (rho t).
// Three times as many rows are undecided (1-4 % of a residual stage instead of 0.3-1.5 %), a third of the matrix
// instructions and half of the staged operands are left.  A value beyond the range of binary16 makes dx
// infinite, and the row is listed; elements below its normal range count as if they were flushed.
// The line lies where the matrix instructions outweigh the undecided rows (three parts -> one product,
// encode of 400,000 rows): k = 256: sd = 32 311 -> 328 us (8 blocks), 48 199 -> 193, 64 239 -> 207 (4 blocks),
// 128 110 -> 88, 256 203 -> 153 (1 block); k = 64: sd = 64 70 -> 74 (2 blocks), 128 65 -> 64; k = 32: sd = 256
// 125 -> 117.
// t: where most centroids are as long as the rows (a random codebook) 0.35 leaves 6.3 % of the rows undecided and
// 0.6 4.5 %, where they are short (a late residual stage) 2 and 3 %.
constexpr float kWideRho = 2.0e-4f, kWideHalfT = 0.6f;
constexpr float kWideTwo = 2.1f, kWideHalfTwo = 2.01f;  // both shares twice, and the roundings of x2, pen and the bound itself
inline bool wide_half(int sd, int nb) { return sd >= 64 && sd * nb >= 512; }
constexpr int kWideCentreMax = 2048;  // widest column block whose centre is staged in LDS

struct MfmaWideBfTables {
    const u32x4 *atab;     // [m][ceil(sd/16)][nb][2][64]  ah, then al, of the lane's eight dimensions
                           // (HALF: [m][ceil(sd/16)][nb][64])
    const float *c2perm;   // [m][nb][2][16]  ||c - mu||^2 less the centroid's share of the error bound
    const float *pen;      // [m][nb * 32]  that share
    const float *blockmax; // [m][nb]  largest ||c - mu||^2 per block of 32 centroids (NaN if any is NaN)
    const float *mu;       // [m][sd]  centre of every column block: mean of its centroids
    const int *shifted;    // [m]  0: the centre is not used
    const float *sigma;    // [m]  HALF: the scale
    uint32_t *list;        // undecided pairs (row * m + s) for the exact kernel over all centroids
    uint32_t *list_count;  // [0] entries of list, [1] entries of pairs
    uint2 *pairs;          // undecided pairs with only two candidates: {row * m + s, c1 | c2 << 8}
    u32x4 *masks;          // k_assign_mfma_wide_res: [mask_cap][2] the candidates of an entry of list (candidate_bit)
    uint32_t mask_cap;
    int nb;
    int sd;
    float kappa;           // COS: error-bound coefficient on ||x||
    float row_share;       // else: the rows' share of the bound of two candidates, per unit of ||x - mu||^2,
    float dx_share;        // HALF: and per unit of dx^2,
    float lift;            // what is added to the scores so that they are positive, likewise,
    float rel;             // and the tag and the reference's rounding, per unit of the score
};

// One workgroup per (column block s, block b of 32 centroids): thread (i, g) = (tid % 32, tid / 32)
// writes the chunks kc = g, g + 8, ... of centroid 32 b + i and sums their share of ||c||^2; the
// eight shares are added in g order.  blockmax[s][b] = largest ||c||^2 of the block (NaN stays).
// mu[s][t] = mean over the k <= 256 centroids of column block s (sum of c / 256, then * 256 / k:
// no overflow).  Rows and centroids are scored relative to it, as in k_mfma8_prep, when that
// shrinks the norms the error bound is proportional to: k_mfma_wide_bf_prep sets shifted[s] = 0
// and ignores the centre if ||mu||^2 is no more than a quarter of the mean ||c||^2 (or the block
// is wider than kWideCentreMax), and the assignment kernel then skips the subtraction.  Grid (m, ceil(sd / 32)); thread (i, g) =
// (tid % 32, tid / 32) adds the centroids g, g + 8, ... of dimension 32 y + i; norms[s][y] =
// this slice's share of {||mu||^2, mean ||c||^2}.
static __global__ void __launch_bounds__(256) k_block_centres(const float *__restrict__ cb, int k, int sd,
                                                              float *__restrict__ mu, float2 *__restrict__ norms) {
    const int s = blockIdx.x, y = blockIdx.y;
    const int i = threadIdx.x & 31, g = threadIdx.x >> 5;
    const int t = 32 * y + i;
    __shared__ float part[2][8][32];
    float acc = 0.0f, sq = 0.0f;
    if (t < sd) {
        const float *c = cb + (size_t)s * k * sd + t;
        float v[32];  // k <= 256: all of the thread's loads are in flight together
#pragma unroll
        for (int u = 0; u < 32; ++u) {
            const int j = g + 8 * u;
            v[u] = c[(size_t)(j < k ? j : 0) * sd];
        }
#pragma unroll
        for (int u = 0; u < 32; ++u) {
            const float w = (g + 8 * u < k) ? v[u] * 0.00390625f : 0.0f;
            acc += w;
            sq = __builtin_fmaf(w, w, sq);
        }
    }
    part[0][g][i] = acc;
    part[1][g][i] = sq;
    __syncthreads();
    if (g == 0) {
        float a = 0.0f, q = 0.0f;
#pragma unroll
        for (int u = 0; u < 8; ++u) {
            a += part[0][u][i];
            q += part[1][u][i];
        }
        const float ctr = a * (256.0f / (float)k);
        if (t < sd) mu[(size_t)s * sd + t] = ctr;
        float mm = (t < sd) ? ctr * ctr : 0.0f, cc = q * (65536.0f / (float)k);
#pragma unroll
        for (int off = 16; off > 0; off >>= 1) {
            mm += __shfl_xor(mm, off);
            cc += __shfl_xor(cc, off);
        }
        if (i == 0) norms[(size_t)s * gridDim.y + y] = make_float2(mm, cc);
    }
}

// COS: the operands of the centroids divided by their norms (cnorm), no centre, no ||c||^2; blockmax is 0,
// or NaN where a norm is outside the range that the scores can decide (see cos_normalise).
// CENTRE: up to wide_own_centre's size every workgroup makes the centre itself (the same sums in the same order
// in each; 32 loads per thread in flight) instead of waiting for a launch of k_block_centres: encode of 1,500 x
// 8 blocks of 32, k = 256: 18.2 -> 16.7 us, 400,000 rows 308-313 us either way.
inline bool wide_own_centre(int k, int sd) { return sd <= 256 && k <= 32 * (256 / sd); }
template <bool COS = false, bool HALF = false, bool CENTRE = false>
static __global__ void __launch_bounds__(256) k_mfma_wide_bf_prep(const float *__restrict__ cb,
                                                                  float *__restrict__ mu,
                                                                  const float2 *__restrict__ norms,
                                                                  int *__restrict__ shifted, int m, int k, int nb,
                                                                  int sd, u32x4 *__restrict__ atab,
                                                                  float *__restrict__ c2perm,
                                                                  float *__restrict__ blockmax,
                                                                  uint32_t *__restrict__ list_count,
                                                                  float *__restrict__ pen, float pen_c2,
                                                                  float *__restrict__ sigma, float pen_dc,
                                                                  int count_step,
                                                                  const float *__restrict__ cnorm = nullptr) {
    const int s = blockIdx.x, b = blockIdx.y;
    const int i = threadIdx.x & 31, g = threadIdx.x >> 5;
    const int j = b * 32 + i;
    const int npair = (sd + 15) / 16;
    __shared__ float part[8][32];
    __shared__ float part_dc[8][32];
    // the same decision in every workgroup of the column block (same values, same order)
    float mm = 0.0f, cc = 0.0f;
    __shared__ __attribute__((aligned(16))) float own_mu[CENTRE ? 256 : 4];
    if constexpr (CENTRE) {
        __shared__ float sums[2][256], red[2];
        const int G = 256 / sd, t = threadIdx.x % sd, q = threadIdx.x / sd;  // centroids q, q + G, ... of dimension t
        float a = 0.0f, sq = 0.0f;
        const float *col = cb + (size_t)s * k * sd + t;
        float v[32];
#pragma unroll
        for (int u = 0; u < 32; ++u) v[u] = col[(size_t)(q + G * u < k ? q + G * u : 0) * sd];
#pragma unroll
        for (int u = 0; u < 32; ++u) {
            const float w = (q < G && q + G * u < k) ? v[u] * 0.00390625f : 0.0f;
            a += w;
            sq = __builtin_fmaf(w, w, sq);
        }
        sums[0][threadIdx.x] = a;
        sums[1][threadIdx.x] = sq;
        __syncthreads();
        if ((int)threadIdx.x < sd) {
            a = 0.0f;
            sq = 0.0f;
            for (int u = 0; u < G; ++u) {
                a += sums[0][u * sd + t];
                sq += sums[1][u * sd + t];
            }
            const float ctr = a * (256.0f / (float)k);
            own_mu[t] = ctr;
            if (b == 0) mu[(size_t)s * sd + t] = ctr;
            sums[1][t] = sq;  // (only this thread has read it)
        }
        __syncthreads();
        if (threadIdx.x < 64) {
            for (int u = threadIdx.x; u < sd; u += 64) {
                mm = __builtin_fmaf(own_mu[u], own_mu[u], mm);
                cc += sums[1][u];
            }
#pragma unroll
            for (int off = 32; off > 0; off >>= 1) {
                mm += __shfl_xor(mm, off);
                cc += __shfl_xor(cc, off);
            }
            if (threadIdx.x == 0) {
                red[0] = mm;
                red[1] = cc * (65536.0f / (float)k);
            }
        }
        __syncthreads();
        mm = red[0];
        cc = red[1];
    }
    for (int y = 0; y < (COS || CENTRE ? 0 : (sd + 31) / 32); ++y) {
        const float2 v = norms[(size_t)s * ((sd + 31) / 32) + y];
        mm += v.x;
        cc += v.y;
    }
    const float nc = COS ? cnorm[(size_t)s * k + (j < k ? j : 0)] : 1.0f;
    const float scale = nc == 0.0f ? 0.0f : -2.0f * (1.0f / nc);
    const bool on = !COS && mm > 0.25f * cc && mm < 1e30f && sd <= kWideCentreMax;  // false for NaN
    float sg = 1.0f;
    if constexpr (HALF) {
        // (1e-6: where mean ||c||^2 and ||mu||^2 cancel, any scale will do)
        const float r2 = on ? fmaxf(cc - mm, 1e-6f * cc) : cc;
        if (r2 > 1e-36f && r2 < 1e36f) sg = ldexpf(1.0f, 5 - (ilogbf(r2) >> 1));
    }
    if (b == 0 && threadIdx.x == 0) {
        shifted[s] = on ? 1 : 0;
        if constexpr (HALF) sigma[s] = sg;
    }
    const float *c = cb + ((size_t)s * k + (j < k ? j : 0)) * sd;
    float p = 0.0f, dcs = 0.0f;
    for (int pr = g; pr < npair; pr += 8) {
        // lane i + 32 h holds the dimensions 16 pr + 8 h .. + 7 (zeros past the block's width): 16
        // bytes of high parts, then, 64 entries on, 16 bytes of low parts, each the operand of a
        // matrix instruction as it lies in LDS
        u32x4 *dst = atab + (((size_t)s * npair + pr) * nb + b) * (HALF ? 64 : 128);
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const int d0 = 16 * pr + 8 * h;
            const bool in = d0 < sd;  // sd is a multiple of 8
            const int dc = in ? d0 : 0;
            const float4 v0 = *reinterpret_cast<const float4 *>(c + dc);
            const float4 v1 = *reinterpret_cast<const float4 *>(c + dc + 4);
            float4 u0 = make_float4(0.f, 0.f, 0.f, 0.f), u1 = u0;
            if (on) {
                const float *ctr = CENTRE ? own_mu : mu + (size_t)s * sd;
                u0 = *reinterpret_cast<const float4 *>(ctr + dc);
                u1 = *reinterpret_cast<const float4 *>(ctr + dc + 4);
            }
            float cv[8] = {v0.x - u0.x, v0.y - u0.y, v0.z - u0.z, v0.w - u0.w,
                           v1.x - u1.x, v1.y - u1.y, v1.z - u1.z, v1.w - u1.w};
            if constexpr (HALF) {
                f16x8 hv;
#pragma unroll
                for (int e = 0; e < 8; ++e) {
                    const float x = in ? cv[e] * sg : 0.0f;
                    p = __builtin_fmaf(x, x, p);
                    const float a = (j < k) ? -2.0f * x : 0.0f;
                    hv[e] = (_Float16)a;
                    if (fabsf((float)hv[e]) < 6.103515625e-05f) hv[e] = (_Float16)0.0f;
                    const float d = a - (float)hv[e];
                    dcs = __builtin_fmaf(d, d, dcs);
                }
                dst[32 * h + i] = __builtin_bit_cast(u32x4, hv);
                continue;
            }
            uint32_t hw[4], lw[4];  // packed pairs of the high and low parts
#pragma unroll
            for (int w = 0; w < 4; ++w) {
                uint32_t hb[2], lb[2];
#pragma unroll
                for (int e = 0; e < 2; ++e) {
                    const float x = in ? cv[2 * w + e] : 0.0f;
                    p = __builtin_fmaf(x, x, p);
                    const float a = (j < k) ? (COS ? scale : -2.0f) * x : 0.0f;
                    hb[e] = bf16_rne_bits(a);
                    lb[e] = bf16_rne_bits(a - bf16_bits_to_float(hb[e]));
                }
                hw[w] = hb[0] | (hb[1] << 16);
                lw[w] = lb[0] | (lb[1] << 16);
            }
            dst[32 * h + i] = u32x4{hw[0], hw[1], hw[2], hw[3]};
            dst[64 + 32 * h + i] = u32x4{lw[0], lw[1], lw[2], lw[3]};
        }
    }
    part[g][i] = p;
    if constexpr (HALF) part_dc[g][i] = dcs;
    __syncthreads();
    if (g == 0) {
        float c2 = 0.0f;
#pragma unroll
        for (int q = 0; q < 8; ++q) c2 = c2 + part[q][i];
        dcs = 0.0f;
        if constexpr (HALF) {
#pragma unroll
            for (int q = 0; q < 8; ++q) dcs = dcs + part_dc[q][i];
            dcs *= 0.25f;  // (the operand is -2 c)
        }
        if constexpr (COS) c2 = nc == 0.0f || (nc >= 1e-15f && nc <= 1e15f) ? 0.0f : __builtin_nanf("");
        float mx = c2;
        const float share = COS ? 0.0f : pen_c2 * c2 + (HALF ? pen_dc * dcs : 0.0f);
        c2 = COS ? 0.0f : c2 - share;
        if (j >= k) {
            c2 = kPadScore;
            mx = 0.0f;
        }
        pen[((size_t)s * nb + b) * 32 + i] = share;
        const int hh = (i / 4) % 2, v = (i / 8) * 4 + i % 4;
        c2perm[(((size_t)s * nb + b) * 2 + hh) * 16 + v] = c2;
#pragma unroll
        for (int off = 16; off > 0; off >>= 1) {
            const float o = __shfl_xor(mx, off);
            mx = (mx == mx && o == o) ? fmaxf(mx, o) : __builtin_nanf("");
        }
        if (i == 0) blockmax[(size_t)s * nb + b] = mx;
        if (b == 0 && i < 2) list_count[(m - 1 - s) * count_step + i] = 0;  // (step 0: one pair for all column blocks)
    }
}

// LDS writes of this wave done, then the workgroup barrier; vector-memory loads stay in flight
// (__syncthreads would wait for the prefetches as well).
__device__ __forceinline__ void lds_barrier() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

// HALF: the row operands of 32 dimensions, a lane's 8 of each 16 (from d0 and d0 + 16; zeros past the
// width: the surplus loads repeat the row's first pieces, and a factor of zero takes them out).  mu: -mu sigma,
// zeros up to a multiple of 32.
__device__ __forceinline__ void wide_round(const float4 (&p)[4], int d0, int sd, bool shifted, const float *mu, float sg,
                                           f16x8 (&b)[2], float &x2, float &dx2) {
    using h2 = _Float16 __attribute__((ext_vector_type(2)));
    using f2 = float __attribute__((ext_vector_type(2)));
#pragma unroll
    for (int q = 0; q < 2; ++q) {
        const float sq = d0 + 16 * q < sd ? sg : 0.0f;
        float xv[8] = {p[2 * q].x, p[2 * q].y, p[2 * q].z, p[2 * q].w,
                       p[2 * q + 1].x, p[2 * q + 1].y, p[2 * q + 1].z, p[2 * q + 1].w};
        if (shifted) {  // x sigma - mu sigma in one rounding
            const float4 m0 = *reinterpret_cast<const float4 *>(mu + d0 + 16 * q);
            const float4 m1 = *reinterpret_cast<const float4 *>(mu + d0 + 16 * q + 4);
            const float mv[8] = {m0.x, m0.y, m0.z, m0.w, m1.x, m1.y, m1.z, m1.w};
#pragma unroll
            for (int u = 0; u < 8; ++u) xv[u] = __builtin_fmaf(xv[u], sq, mv[u]);
        } else {
#pragma unroll
            for (int u = 0; u < 8; ++u) xv[u] *= sq;
        }
        uint32_t w[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) {
            w[u] = __builtin_bit_cast(uint32_t, __builtin_convertvector((f2{xv[2 * u], xv[2 * u + 1]}), h2));
            float dl, dh;  // x - xh: one instruction each that reads a half of the pair
            asm("v_fma_mix_f32 %0, %1, -1.0, %2 op_sel_hi:[1,0,0]" : "=v"(dl) : "v"(w[u]), "v"(xv[2 * u]));
            asm("v_fma_mix_f32 %0, %1, -1.0, %2 op_sel:[1,0,0] op_sel_hi:[1,0,0]" : "=v"(dh) : "v"(w[u]), "v"(xv[2 * u + 1]));
            x2 = __builtin_fmaf(xv[2 * u], xv[2 * u], x2);
            x2 = __builtin_fmaf(xv[2 * u + 1], xv[2 * u + 1], x2);
            dx2 = __builtin_fmaf(dl, dl, dx2);
            dx2 = __builtin_fmaf(dh, dh, dx2);
        }
        b[q] = __builtin_bit_cast(f16x8, u32x4{w[0], w[1], w[2], w[3]});
    }
}

// grid (ceil(n/128), m); 256 threads = 4 waves, one tile of 32 rows each against every centroid.
// NB = tiles of 32 centroids (tb.nb), a template parameter so that the chains of matrix
// instructions are straight-line code.
// PEND (one column block): the rows are a residual whose update by the previous stage's codebook is
// still pending, x[i] -= pend_cb[pend_codes[i]] (src/rvq.rs:124-129 in a fit, 200-202 in an encode).
// A workgroup first updates its own 128 rows — whole rows per wave instruction, one f32 subtraction
// per element, as the separate pass would; in place, or from the rows of a.pend_src into a.x — and
// then scores them as any other rows, which it now reads from the cache levels it has just written
// through.  No other workgroup reads or writes these rows.
// COS: cosine distance (see cos_normalise): the scores are P - 2 x.c/|c| with P = 2.01 |x|, the bound is in
// units of |x|.
template <bool LBG, int NB, bool PEND = false, bool COS = false, bool HALF = false>
__global__ void __launch_bounds__(256, 2) k_assign_mfma_wide_bf(AssignArgs a, MfmaWideBfTables tb) {
    constexpr int NBMAX = 8;
    __shared__ u32x4 lds_a[2][NBMAX * 128];  // 2 stages x 16 dimensions x 256 centroids x {high, low}: 2 x 16 KB
    __shared__ float lds_c2[NBMAX * 32];
    __shared__ float lds_pen[COS ? 1 : NBMAX * 32];
    __shared__ float lds_mu[kWideCentreMax];
    __shared__ uint32_t wg_list[128];
    __shared__ uint2 wg_pairs[128];
    __shared__ uint32_t wg_count, wg_base, wg_pcount, wg_pbase;
    const int s = blockIdx.y;
    if constexpr (LBG) {
        if (block_done(a, s)) return;
    }
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int r = lane & 31, h = lane >> 5;
    constexpr int nb = NB;
    const int sd = tb.sd, npair = (sd + 15) / 16;
    const u32x4 *ag = tb.atab + (size_t)s * npair * nb * (HALF ? 64 : 128);
    const int pair16 = nb * 128;  // 16-byte pieces per 16 dimensions (HALF: per 32)
    const int total16 = npair * nb * (HALF ? 64 : 128);
    const float sg = HALF ? tb.sigma[s] : 1.0f;
    for (int i = threadIdx.x; i < nb * 32; i += 256) lds_c2[i] = tb.c2perm[(size_t)s * nb * 32 + i];
    if constexpr (!COS)
        for (int i = threadIdx.x; i < nb * 32; i += 256) lds_pen[i] = tb.pen[(size_t)s * nb * 32 + i];
    for (int i = threadIdx.x; i < pair16; i += 256) lds_a[0][i] = ag[i < total16 ? i : total16 - 1];
    if (threadIdx.x == 0) {
        wg_count = 0;
        wg_pcount = 0;
    }
    if (tb.shifted[s] != 0)
        for (int i = threadIdx.x; i < (HALF ? (sd + 31) & ~31 : sd); i += 256) {
            const float c = tb.mu[(size_t)s * sd + (i < sd ? i : 0)];
            lds_mu[i] = !HALF ? c : i < sd ? -(c * sg) : 0.0f;
        }
    if constexpr (PEND) {
        const int64_t row0 = (int64_t)blockIdx.x * 128;
        const int nrows = a.n - row0 < 128 ? (int)(a.n - row0) : 128;
        float *xw = const_cast<float *>(a.x) + row0 * a.ld;
        const float *xr = a.pend_src ? a.pend_src + row0 * a.pend_src_ld : xw;
        const int64_t xr_ld = a.pend_src ? a.pend_src_ld : a.ld;
        const uint8_t *pc = a.pend_codes + row0;
        const int per_row = sd / 4, total = nrows * per_row;  // 16-byte pieces
        constexpr int B = 8;  // pieces of a thread in flight together
        for (int i0 = threadIdx.x; i0 < total; i0 += 256 * B) {
            float4 v[B], c[B];
#pragma unroll
            for (int u = 0; u < B; ++u) {
                const int i = i0 + 256 * u < total ? i0 + 256 * u : i0;
                const int rr = i / per_row, cc = i - rr * per_row;
                v[u] = *reinterpret_cast<const float4 *>(xr + (int64_t)rr * xr_ld + 4 * cc);
                c[u] = *reinterpret_cast<const float4 *>(a.pend_cb + (size_t)pc[rr] * sd + 4 * cc);
            }
#pragma unroll
            for (int u = 0; u < B; ++u) {
                const int i = i0 + 256 * u;
                if (i < total) {
                    const int rr = i / per_row, cc = i - rr * per_row;
                    *reinterpret_cast<float4 *>(xw + (int64_t)rr * a.ld + 4 * cc) =
                        make_float4(v[u].x - c[u].x, v[u].y - c[u].y, v[u].z - c[u].z, v[u].w - c[u].w);
                }
            }
        }
    }
    __syncthreads();  // (PEND: the updated rows are visible to every wave of the workgroup)

    const int64_t row = (int64_t)blockIdx.x * 128 + wave * 32 + r;
    const bool valid = row < a.n;
    // the workgroup's first row is a scalar base, the lane's row a 32-bit byte offset from it (the
    // host keeps 128 rows below 2^31 bytes); a row past the end reads the workgroup's first row
    const char *xwg = reinterpret_cast<const char *>(a.x + (int64_t)blockIdx.x * 128 * a.ld + (int64_t)s * sd);
    const uint32_t xlane = valid ? 4u * (uint32_t)(wave * 32 + r) * (uint32_t)a.ld : 0u;
    auto row_piece = [&](int d) { return *reinterpret_cast<const float4 *>(xwg + (xlane + 4u * (uint32_t)d)); };
    const bool shifted = tb.shifted[s] != 0;  // uniform
    // the accumulators start at ||c - mu||^2 less the centroid's share of the bound; ||x - mu||^2, the same
    // in every score of a row, is summed on the side and added, a little enlarged, before the selection
    // (a score is then positive, and its bits order as an integer)
    floatx16 acc[NB];
#pragma unroll
    for (int b = 0; b < NB; ++b)
#pragma unroll
        for (int v = 0; v < 16; ++v) acc[b][v] = lds_c2[(b * 2 + h) * 16 + v];
    // Loads are unconditional (a row past the end reads row 0 and is never stored; pieces past
    // the block's width are clamped and zeroed): loads under a branch make the compiler wait for
    // every outstanding load at each use instead of counting them.
    // This half's 8 of the 16 dimensions of a stage: 16 pr + 8 h .. + 7.
    auto piece = [&](int pr) { return 16 * pr + 8 * h < sd ? 16 * pr + 8 * h : 0; };
    float x2 = 0.0f, dx2 = 0.0f;
    if constexpr (HALF) {
        // A stage is 32 dimensions in two steps of 16: whole 128-byte lines of a row per stage, one barrier
        // per 2 NB matrix instructions; a last step past the width is left out.
        const int nst = (npair + 1) / 2;
        auto fetch = [&](int st, float4(&p)[4]) {
#pragma unroll
            for (int q = 0; q < 2; ++q) {
                const int d = piece(2 * st + q);
                p[2 * q] = row_piece(d);
                p[2 * q + 1] = row_piece(d + 4);
            }
        };
        auto halves = [&](int st, const float4(&p)[4], f16x8(&b)[2]) {
            wide_round(p, 32 * st + 8 * h, sd, shifted, lds_mu, sg, b, x2, dx2);
        };
        float4 xn[4], xf[4];
        f16x8 b[2], bn[2];
        fetch(0, xn);
        fetch(1 < nst ? 1 : 0, xf);
        halves(0, xn, b);
#pragma unroll
        for (int q = 0; q < 4; ++q) xn[q] = xf[q];
        fetch(2 < nst ? 2 : nst - 1, xf);
        for (int st = 0; st < nst; ++st) {
            const int cur = st & 1;
            const bool more = st + 1 < nst;
            u32x4 pre[4];
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                const uint32_t i = (uint32_t)((st + 1) * pair16) + threadIdx.x + 256u * (uint32_t)q;
                const uint32_t ic = i < (uint32_t)total16 ? i : (uint32_t)total16 - 1u;
                pre[q] = *reinterpret_cast<const u32x4 *>(reinterpret_cast<const char *>(ag) + 16u * ic);
            }
            auto step = [&](int q, const f16x8 &bq) {
#pragma unroll
                for (int b0 = 0; b0 < NB; b0 += 4) {
                    u32x4 ah[4];
#pragma unroll
                    for (int c = 0; c < 4; ++c)
                        if (b0 + c < NB) ah[c] = lds_a[cur][(q * NB + b0 + c) * 64 + lane];
#pragma unroll
                    for (int c = 0; c < 4; ++c)
                        if (b0 + c < NB)
                            acc[b0 + c] = __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(f16x8, ah[c]), bq,
                                                                                acc[b0 + c], 0, 0, 0);
                }
            };
            step(0, b[0]);
            if (more) {
                // the next stage's row operands, behind the first matrix instructions of this stage
                halves(st + 1, xn, bn);
#pragma unroll
                for (int q = 0; q < 4; ++q) xn[q] = xf[q];
                fetch(st + 3 < nst ? st + 3 : nst - 1, xf);
            }
            if (2 * st + 1 < npair) step(1, b[1]);
            b[0] = bn[0];
            b[1] = bn[1];
            if (more) {
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    const int i = threadIdx.x + 256 * q;
                    if (i < pair16) lds_a[cur ^ 1][i] = pre[q];
                }
            }
            lds_barrier();
        }
        dx2 += __shfl_xor(dx2, 32);
    } else {
        float4 xn0 = row_piece(piece(0));  // the next piece of the row
        float4 xn1 = row_piece(piece(0) + 4);
        const int second = npair > 1 ? 1 : 0;
        float4 xf0 = row_piece(piece(second));  // and the one after it
        float4 xf1 = row_piece(piece(second) + 4);
        // The row operands of a stage: this half's 8 dimensions relative to the centre, their share of
        // ||x - mu||^2, and their high and low bf16 parts.
        auto split = [&](int st, const float4 &p0, const float4 &p1, u32x4 &bh, u32x4 &bl) {
            float xv[8] = {p0.x, p0.y, p0.z, p0.w, p1.x, p1.y, p1.z, p1.w};
            if (shifted) {
                const float4 m0 = *reinterpret_cast<const float4 *>(lds_mu + piece(st));
                const float4 m1 = *reinterpret_cast<const float4 *>(lds_mu + piece(st) + 4);
                xv[0] -= m0.x;
                xv[1] -= m0.y;
                xv[2] -= m0.z;
                xv[3] -= m0.w;
                xv[4] -= m1.x;
                xv[5] -= m1.y;
                xv[6] -= m1.z;
                xv[7] -= m1.w;
            }
            if (st == npair - 1 && (sd & 8) != 0) {  // uniform: a width that is an odd multiple of 8 ends in the lower half
                if (h != 0) {
    #pragma unroll
                    for (int u = 0; u < 8; ++u) xv[u] = 0.0f;
                }
            }
            uint32_t hp[4], lp[4];
    #pragma unroll
            for (int u = 0; u < 4; ++u) {
                x2 = __builtin_fmaf(xv[2 * u], xv[2 * u], x2);
                x2 = __builtin_fmaf(xv[2 * u + 1], xv[2 * u + 1], x2);
                hp[u] = bf16_pack2(xv[2 * u], xv[2 * u + 1]);
                lp[u] = bf16_pack2(xv[2 * u] - __uint_as_float(hp[u] << 16), xv[2 * u + 1] - __uint_as_float(hp[u] & 0xffff0000u));
            }
            bh = u32x4{hp[0], hp[1], hp[2], hp[3]};
            bl = u32x4{lp[0], lp[1], lp[2], lp[3]};
        };
        // A stage is 16 dimensions: with the high and low parts of the centroid operand (ah, al) and of
        // the row operand (xh, xl), three matrix instructions per tile of 32 centroids,
        //   ah . xh + al . xh + ah . xl,
        // every contraction slot of each in use; one barrier per 3 NB matrix instructions of a wave.
        // The row operands of stage st + 1 are made while the matrix instructions of stage st run: a
        // matrix instruction holds back the vector instructions of the other waves of its SIMD, but
        // independent vector instructions of its own wave issue in its shadow.
        u32x4 bh, bl;
        split(0, xn0, xn1, bh, bl);
        xn0 = xf0;
        xn1 = xf1;
        {
            const int nx = 2 < npair ? 2 : npair - 1;
            xf0 = row_piece(piece(nx));
            xf1 = row_piece(piece(nx) + 4);
        }
        for (int st = 0; st < npair; ++st) {
            const int cur = st & 1;
            const bool more = st + 1 < npair;
            // the A operands of the next stage: into registers now, into LDS at the end of this stage
            u32x4 pre[4];
    #pragma unroll
            for (int q = 0; q < 4; ++q) {
                const uint32_t i = (uint32_t)((st + 1) * pair16) + threadIdx.x + 256u * (uint32_t)q;
                const uint32_t ic = i < (uint32_t)total16 ? i : (uint32_t)total16 - 1u;
                pre[q] = *reinterpret_cast<const u32x4 *>(reinterpret_cast<const char *>(ag) + 16u * ic);
            }
            // The stage's centroid operands are read from LDS four tiles (one group) at a time.
            constexpr int NG = (NB + 3) / 4;  // groups of four centroid tiles
            u32x4 nbh = bh, nbl = bl;
    #pragma unroll
            for (int g = 0; g < NG; ++g) {
                u32x4 ah[4], al[4];
    #pragma unroll
                for (int c = 0; c < 4; ++c) {
                    const int b = 4 * g + c < nb ? 4 * g + c : nb - 1;  // past the last block: read it, not multiplied
                    ah[c] = lds_a[cur][b * 128 + lane];
                    al[c] = lds_a[cur][b * 128 + 64 + lane];
                }
                // the three dependent instructions of a tile are three others apart
    #pragma unroll
                for (int c = 0; c < 4; ++c)
                    if (4 * g + c < nb)
                        acc[4 * g + c] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(
                            __builtin_bit_cast(bf16x8, ah[c]), __builtin_bit_cast(bf16x8, bh), acc[4 * g + c], 0, 0, 0);
                if (g == 0 && more) {
                    // next stage's row operands, behind the first matrix instructions of this stage
                    split(st + 1, xn0, xn1, nbh, nbl);
                    const int nx = st + 3 < npair ? st + 3 : npair - 1;
                    xn0 = xf0;
                    xn1 = xf1;
                    xf0 = row_piece(piece(nx));
                    xf1 = row_piece(piece(nx) + 4);
                }
    #pragma unroll
                for (int c = 0; c < 4; ++c)
                    if (4 * g + c < nb)
                        acc[4 * g + c] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(
                            __builtin_bit_cast(bf16x8, al[c]), __builtin_bit_cast(bf16x8, bh), acc[4 * g + c], 0, 0, 0);
    #pragma unroll
                for (int c = 0; c < 4; ++c)
                    if (4 * g + c < nb)
                        acc[4 * g + c] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(
                            __builtin_bit_cast(bf16x8, ah[c]), __builtin_bit_cast(bf16x8, bl), acc[4 * g + c], 0, 0, 0);
            }
            bh = nbh;
            bl = nbl;
            if (more) {
    #pragma unroll
                for (int q = 0; q < 4; ++q) {
                    const int i = threadIdx.x + 256 * q;
                    if (i < pair16) lds_a[cur ^ 1][i] = pre[q];
                }
            }
            lds_barrier();
        }
    }
    x2 += __shfl_xor(x2, 32);  // both halves' shares of ||x - mu||^2
    const float nx = COS ? __builtin_amdgcn_sqrtf(x2) : 0.0f;
    const float lifted = COS ? 2.01f * nx : HALF ? tb.lift * x2 + 1.0f : tb.lift * x2;
    // the three smallest scores of the row, the index in the low 8 bits (one v_and_or per score; the
    // tag leaves out the lane half, bit 2, so it is the same in every lane: a scalar operand)
    int m1 = 0x7f800000, m2 = 0x7f800000, m3 = 0x7f800000;
    const uint32_t keep = opaque_vgpr(0xFFFFFF00u);
#pragma unroll
    for (int b = 0; b < NB; ++b) {
#pragma unroll
        for (int v = 0; v < 16; v += 4) {
            int key[4];
#pragma unroll
            for (int u = 0; u < 4; ++u)
                key[u] = pack_tag(acc[b][v + u] + lifted, keep, (uint32_t)(32 * b + 8 * (v / 4) + u));
            top3_push4(m1, m2, m3, key[0], key[1], key[2], key[3]);
        }
    }
    {
        m1 |= 4 * h;
        m2 |= 4 * h;
        const int o1 = __shfl_xor(m1, 32), o2 = __shfl_xor(m2, 32), o3 = __shfl_xor(m3, 32);
        top3_push4(m1, m2, m3, o1, o2, o3, 0x7f800000);
    }
    const uint32_t i1 = (uint32_t)m1 & 0xFFu, i2 = (uint32_t)m2 & 0xFFu;
    if (h == 0) {
        float mc2 = 0.0f;  // largest ||c||^2 of the column block; a NaN stays
        for (int b = 0; b < nb; ++b) {
            const float o = tb.blockmax[(size_t)s * nb + b];
            mc2 = (mc2 == mc2 && o == o) ? fmaxf(mc2, o) : __builtin_nanf("");
        }
        const float s1 = __int_as_float(m1), s2 = __int_as_float(m2), s3 = __int_as_float(m3);
        if (valid) {
            const float bound = (COS ? nx : x2) + mc2;
            const bool finite = (bound < (COS ? 1e15f : 1e29f)) && (!COS || bound > 1e-15f) && (s1 < 1e29f);  // false for NaN
            // (1e-32: what products below the smallest normal number can lose)
            const float slack = COS ? tb.kappa * bound : tb.row_share * x2 + (HALF ? tb.dx_share * (dx2 + (float)sd * 0x1p-28f) : 0.0f) +
                                          (HALF ? kWideHalfTwo : kWideTwo) * lds_pen[COS ? 0 : i1] + 1e-32f;
            const float rel = COS ? 6.103515625e-05f : tb.rel;
            // the smallest exact distance is the best-scored centroid's when the second score is
            // further away than the error bound ...
            const bool sure = finite && (s2 - s1) > rel * fabsf(s2) + slack;
            // ... and one of the two best-scored centroids' when the third score is
            const bool two = finite && (s2 < 1e29f) && (s3 - s1) > rel * fabsf(s3) + slack;
            if (sure) {
                const uint8_t code = (uint8_t)i1;
                if constexpr (LBG) {
                    uint8_t *pc = a.codes + (size_t)s * a.n + row;
                    if (*pc != code) {
                        *pc = code;
                        mark_changed(a.changed + s);
                    }
                } else {
                    a.codes[row * a.m + s] = code;
                }
            } else if (two) {
                wg_pairs[atomicAdd(&wg_pcount, 1u)] = make_uint2((uint32_t)(row * a.m + s), i1 | (i2 << 8));
            } else {
                wg_list[atomicAdd(&wg_count, 1u)] = (uint32_t)(row * a.m + s);
            }
        }
    }
    __syncthreads();
    const uint32_t cnt = wg_count, pcnt = wg_pcount;
    if (cnt == 0 && pcnt == 0) return;
    if (threadIdx.x == 0) {
        if (cnt) wg_base = atomicAdd(tb.list_count, cnt);
        if (pcnt) wg_pbase = atomicAdd(tb.list_count + 1, pcnt);
    }
    __syncthreads();
    for (uint32_t i = threadIdx.x; i < cnt; i += 256) tb.list[wg_base + i] = wg_list[i];
    for (uint32_t i = threadIdx.x; i < pcnt; i += 256) tb.pairs[wg_pbase + i] = wg_pairs[i];
}


// The same scores and decisions (HALF) where the operands of a whole column block fit LDS: one workgroup of
// eight waves per compute unit keeps them (128 KB at 256 x 256) and walks over tiles of 32 rows, each wave on
// its own.  No barrier and no operand fetch in the loop, so nothing but the rows is in flight and the
// prefetch, three stages of 32 dimensions ahead and on across the tiles, is never drained (loads return in
// order: in the staged kernel the wait for the next operands is one for the rows fetched before them too).
// HBM-bound: 1,000,000 x 256, k = 256: 238 us = 4.3 TB/s, where the staged kernel takes 330 (vector ALU and
// matrix cores busy for half of its cycles, the rest waits).  From two tiles per wave on: 60,000 rows of 256
// take 38 us staged, 39.5 resident (256 workgroups fill 128 KB of LDS for one tile per wave); 60,000 x 4 of 64
// 47 and 40; 20,000 x 7 of 72 38.5 and 37.5.
constexpr int kWideResThreads = 512;
constexpr int64_t kWideResMinRows = 256 * 8 * 32 * 2;  // rows x column blocks
inline size_t wide_res_lds(int sd, int nb) {
    const size_t npair = (sd + 15) / 16;
    return npair * nb * 1024 + 2 * (size_t)nb * 128 + ((sd + 31) / 32) * 128 + 8 * 64 * sizeof(uint2);
}

template <bool LBG, int NB>
__global__ void __launch_bounds__(kWideResThreads, 2) k_assign_mfma_wide_res(AssignArgs a, MfmaWideBfTables tb) {
    extern __shared__ u32x4 res_a[];  // [npair][NB][64], ||c||^2, pen, mu, the waves' lists
    const int s = blockIdx.y;
    if constexpr (LBG) {
        if (block_done(a, s)) return;
    }
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int r = lane & 31, h = lane >> 5;
    const int sd = tb.sd, npair = (sd + 15) / 16, nst = (npair + 1) / 2, total16 = npair * NB * 64;
    float *lds_c2 = reinterpret_cast<float *>(res_a + total16), *lds_pen = lds_c2 + NB * 32, *lds_mu = lds_pen + NB * 32;
    uint2 *my_pairs = reinterpret_cast<uint2 *>(lds_mu + ((sd + 31) & ~31)) + wave * 64;
    const float sg = tb.sigma[s];
    const bool shifted = tb.shifted[s] != 0;  // uniform
    const u32x4 *ag = tb.atab + (size_t)s * total16;
    for (int i = threadIdx.x; i < total16; i += kWideResThreads) res_a[i] = ag[i];
    for (int i = threadIdx.x; i < NB * 32; i += kWideResThreads) {
        lds_c2[i] = tb.c2perm[(size_t)s * NB * 32 + i];
        lds_pen[i] = tb.pen[(size_t)s * NB * 32 + i];
    }
    for (int i = threadIdx.x; i < ((sd + 31) & ~31); i += kWideResThreads)
        lds_mu[i] = shifted && i < sd ? -(tb.mu[(size_t)s * sd + i] * sg) : 0.0f;
    float mc2 = 0.0f;  // largest ||c||^2 of the column block; a NaN stays
    for (int b = 0; b < NB; ++b) {
        const float o = tb.blockmax[(size_t)s * NB + b];
        mc2 = (mc2 == mc2 && o == o) ? fmaxf(mc2, o) : __builtin_nanf("");
    }
    __syncthreads();

    const int64_t ntiles = (a.n + 31) / 32, step_tiles = (int64_t)gridDim.x * 8;
    // Where some, but less than half, of the waves have a tile in the last round, those tiles lie on all compute units and not
    // eight on a few: encode of 200,000 x 128, k = 256, four stages (3.05 rounds) 337 -> 325 us, 100,000 x 4 blocks of 64 72.5 -> 70.4; a residual
    // fit of 1M x 256 (15.26) the same within 0.5 %.  Beyond, eight neighbouring tiles to a workgroup are the faster ones: 180,000 x 96 (2.75)
    // 1055 against 1068 us; after whole rounds (65,536 to 1,048,576 rows of one to four blocks) both take the same time.
    const int64_t over = ntiles % step_tiles;
    int64_t tile = over != 0 && over * 2 < step_tiles ? (int64_t)wave * gridDim.x + blockIdx.x : (int64_t)blockIdx.x * 8 + wave;
    if (tile >= ntiles) return;  // (no barrier follows)
    const char *xs = reinterpret_cast<const char *>(a.x + (int64_t)s * sd);
    const int64_t tile_bytes = 128 * a.ld;
    auto lane_base = [&](int64_t t) { return t * 32 + r < a.n ? 4u * (uint32_t)r * (uint32_t)a.ld : 0u; };
    auto piece = [&](int pr) { return 16 * pr + 8 * h < sd ? 16 * pr + 8 * h : 0; };
    // where the prefetch is: it runs on into the wave's next tile (and stays on the last one)
    int64_t ptile = tile;
    int pst = 0;
    const char *pbase = xs + ptile * tile_bytes;
    uint32_t plane = lane_base(ptile);
    auto fetch = [&](float4(&p)[4]) {
#pragma unroll
        for (int q = 0; q < 2; ++q) {
            const uint32_t o = plane + 4u * (uint32_t)piece(2 * pst + q);
            p[2 * q] = *reinterpret_cast<const float4 *>(pbase + o);
            p[2 * q + 1] = *reinterpret_cast<const float4 *>(pbase + (o + 16u));
        }
        if (++pst == nst) {
            pst = 0;
            if (ptile + step_tiles < ntiles) ptile += step_tiles;
            pbase = xs + ptile * tile_bytes;
            plane = lane_base(ptile);
        }
    };
    float4 x0[4], x1[4], x3[4];
    f16x8 b[2], bn[2];
    float x2 = 0.0f, dx2 = 0.0f;
    fetch(x0);
    fetch(x1);
    fetch(x3);
    auto next_rows = [&](int st) {  // the operands of a stage; everything behind it moves up
        wide_round(x0, 32 * st + 8 * h, sd, shifted, lds_mu, sg, bn, x2, dx2);
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            x0[q] = x1[q];
            x1[q] = x3[q];
        }
        fetch(x3);
    };
    next_rows(0);
    const uint32_t keep = opaque_vgpr(0xFFFFFF00u);
    uint32_t npairs = 0;  // uniform
    auto flush_pairs = [&]() {
        uint32_t base = 0;
        if (lane == 0) base = atomicAdd(tb.list_count + 1, npairs);
        base = __builtin_amdgcn_readfirstlane(base);
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
        if ((uint32_t)lane < npairs) tb.pairs[base + lane] = my_pairs[lane];
        __builtin_amdgcn_wave_barrier();
        npairs = 0;
    };
    for (; tile < ntiles; tile += step_tiles) {
        const int64_t row = tile * 32 + r;
        const bool valid = row < a.n;
        uint8_t old = 0;
        if constexpr (LBG) old = a.codes[(size_t)s * a.n + (valid ? row : a.n - 1)];
        floatx16 acc[NB];
#pragma unroll
        for (int c = 0; c < NB; ++c)
#pragma unroll
            for (int v = 0; v < 16; ++v) acc[c][v] = lds_c2[(c * 2 + h) * 16 + v];
        float row2 = 0.0f, rowd2 = 0.0f;
        for (int st = 0; st < nst; ++st) {
            b[0] = bn[0];
            b[1] = bn[1];
            auto step = [&](int pr, const f16x8 &bq) {
#pragma unroll
                for (int b0 = 0; b0 < NB; b0 += 4) {
                    u32x4 ah[4];
#pragma unroll
                    for (int c = 0; c < 4; ++c)
                        if (b0 + c < NB) ah[c] = res_a[(pr * NB + b0 + c) * 64 + lane];
#pragma unroll
                    for (int c = 0; c < 4; ++c)
                        if (b0 + c < NB)
                            acc[b0 + c] = __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(f16x8, ah[c]), bq,
                                                                                acc[b0 + c], 0, 0, 0);
                }
            };
            step(2 * st, b[0]);
            // the next stage's row operands (the next tile's first, behind the last stage), in the shadow of
            // the matrix instructions
            const bool last = st + 1 == nst;
            if (last) {
                row2 = x2;
                rowd2 = dx2;
                x2 = 0.0f;
                dx2 = 0.0f;
            }
            next_rows(last ? 0 : st + 1);
            if (2 * st + 1 < npair) step(2 * st + 1, b[1]);
        }
        row2 += __shfl_xor(row2, 32);
        rowd2 += __shfl_xor(rowd2, 32);
        const float lifted = tb.lift * row2 + 1.0f;
        int m1 = 0x7f800000, m2 = 0x7f800000, m3 = 0x7f800000;
#pragma unroll
        for (int c = 0; c < NB; ++c) {
#pragma unroll
            for (int v = 0; v < 16; v += 4) {
                int key[4];
#pragma unroll
                for (int u = 0; u < 4; ++u)
                    key[u] = pack_tag(acc[c][v + u] + lifted, keep, (uint32_t)(32 * c + 8 * (v / 4) + u));
                top3_push4(m1, m2, m3, key[0], key[1], key[2], key[3]);
            }
        }
        m1 |= 4 * h;
        m2 |= 4 * h;
        const int o1 = __shfl_xor(m1, 32), o2 = __shfl_xor(m2, 32), o3 = __shfl_xor(m3, 32);
        top3_push4(m1, m2, m3, o1, o2, o3, 0x7f800000);
        const uint32_t i1 = (uint32_t)m1 & 0xFFu, i2 = (uint32_t)m2 & 0xFFu;
        const float s1 = __int_as_float(m1), s2 = __int_as_float(m2), s3 = __int_as_float(m3);
        const float bound = row2 + mc2;
        const bool finite = (bound < 1e29f) && (s1 < 1e29f);  // false for NaN
        const float slack = tb.row_share * row2 + tb.dx_share * (rowd2 + (float)sd * 0x1p-28f) +
                            kWideHalfTwo * lds_pen[i1] + 1e-32f;
        const bool sure = finite && (s2 - s1) > tb.rel * fabsf(s2) + slack;
        const bool two = finite && (s2 < 1e29f) && (s3 - s1) > tb.rel * fabsf(s3) + slack;
        const bool mine = valid && h == 0;
        if (mine && sure) {
            if constexpr (LBG) {
                if (old != (uint8_t)i1) {
                    a.codes[(size_t)s * a.n + row] = (uint8_t)i1;
                    mark_changed(a.changed + s);
                }
            } else {
                a.codes[row * a.m + s] = (uint8_t)i1;
            }
        }
        const uint64_t pm = __ballot(mine && !sure && two), lm = __ballot(mine && !sure && !two);
        const uint64_t below = ((uint64_t)1 << lane) - 1;
        if (pm) {  // uniform
            if (npairs > 32) flush_pairs();
            if ((pm >> lane) & 1) my_pairs[npairs + __popcll(pm & below)] = make_uint2((uint32_t)(row * a.m + s), i1 | (i2 << 8));
            npairs += (uint32_t)__popcll(pm);
        }
        if (lm) {
            // the candidates: every centroid that is not clear of the best one (2^-14: the tag's bits); for a row or
            // a block that is not finite all of them
            const float least = (s1 + slack) * (1.0f + 2.0f * tb.rel) * 1.00006103515625f;
            uint32_t mk[4] = {0u, 0u, 0u, 0u};
#pragma unroll
            for (int c = 0; c < NB; ++c)
#pragma unroll
                for (int v = 0; v < 16; ++v)
                    mk[c >> 1] |= !(finite && acc[c][v] + lifted > least) ? 1u << (16 * (c & 1) + v) : 0u;
            uint32_t base = 0;
            if (lane == 0) base = atomicAdd(tb.list_count, (uint32_t)__popcll(lm));
            base = __builtin_amdgcn_readfirstlane(base);
            if ((lm >> r) & 1) {
                const uint32_t e = base + (uint32_t)__popcll(lm & (((uint64_t)1 << r) - 1));
                if (h == 0) tb.list[e] = (uint32_t)(row * a.m + s);
                if (e < tb.mask_cap) tb.masks[2 * (size_t)e + h] = u32x4{mk[0], mk[1], mk[2], mk[3]};
            }
        }
    }
    if (npairs) flush_pairs();
}

// ---- what k_assign_mfma_wide_res leaves open ------------------------------------------------------
// Pairs with two candidates, and rows with a mask of candidates (three to a few dozen of the 256), decided by
// distances in the reference's order: a lane per candidate, each its own sequential chain.  The vectors come through LDS
// 32 dimensions at a time, eight lanes per 128-byte segment, the next 32 in flight meanwhile (the pieces' order
// depends on the slot: the lanes' 16-byte reads fall into different banks; 48 KB, three workgroups in a compute unit).  A lane that read its own row and centroid from memory touched 64 lines
// per load instruction and had 64 of them one after the other, and a row that more than two centroids could win was
// compared with all of them: per pass of a residual fit of 1M x 256, k = 256 (15,000-60,000 pairs, 500-4,000 rows) 54 us,
// 20 so, the fit 50.1 -> 47.3 ms.  Bound by the rows from HBM (up to 60 MB; slices of 16 dimensions, or four in flight, the same).
constexpr int kFollowSlots = 96;  // 32 rows and 64 centroids per wave, 32 floats each
constexpr unsigned kFollowPairBlocks = 512, kFollowRowBlocks = 2048;
constexpr uint32_t kFollowMany = 16384;  // rows from which on their candidates may be all centroids for all we know

// Bit of centroid j in an entry's masks: half (j / 4) % 2, then 16 bits per block of 32.
__device__ __forceinline__ bool candidate_bit(const u32x4 *mask, int j) {
    const int c = j >> 5, v = ((j >> 3) & 3) * 4 + (j & 3);
    const uint32_t w = reinterpret_cast<const uint32_t *>(mask + ((j >> 2) & 1))[c >> 1];
    return (w >> (16 * (c & 1) + v)) & 1u;
}

template <bool LBG> __device__ __forceinline__ void store_code(const AssignArgs &a, int64_t row, int s, int code) {
    if constexpr (LBG) {
        uint8_t *p = a.codes + (size_t)s * a.n + row;
        if (*p != (uint8_t)code) {
            *p = (uint8_t)code;
            mark_each_changed(a.changed + s);
        }
    } else {
        a.codes[row * a.m + s] = (uint8_t)code;
    }
}

__device__ __forceinline__ float4 *follow_piece(float *st, int slot, int piece) {
    return reinterpret_cast<float4 *>(st + slot * 32 + 4 * (piece ^ ((slot >> 1) & 7)));
}
// The distance of the row in slot x to the centroid in slot c: acc goes on over 32 dimensions (nd of them) in LDS.
template <int METRIC> __device__ __forceinline__ void follow_slice(float &acc, float *st, int x, int c, int nd) {
#pragma unroll
    for (int p = 0; p < 8; ++p) {
        if (4 * p >= nd) break;  // uniform
        const float4 xv = *follow_piece(st, x, p), cv = *follow_piece(st, c, p);
        wide_step<METRIC>(acc, xv.x, cv.x);
        wide_step<METRIC>(acc, xv.y, cv.y);
        wide_step<METRIC>(acc, xv.z, cv.z);
        wide_step<METRIC>(acc, xv.w, cv.w);
    }
}

template <int METRIC, bool LBG>
__global__ void __launch_bounds__(256) k_wide_follow(AssignArgs a, int sd, const uint32_t *__restrict__ list,
                                                     const uint32_t *__restrict__ counts, const u32x4 *__restrict__ masks,
                                                     uint32_t mask_cap, const uint2 *__restrict__ pairs) {
    static_assert(METRIC == M_SQ || METRIC == M_EUCLID, "squared L2 / Euclidean");
    __shared__ __attribute__((aligned(16))) float stage[4][kFollowSlots * 32];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, sub = lane >> 3, piece = lane & 7;
    float *st = stage[wave];
    const int nsl = (sd + 31) / 32, m = a.m, k = a.k;
    const float inf = __builtin_inff();
    auto at = [&](int sl) { return 32 * sl + 4 * piece < sd ? 32 * sl + 4 * piece : 0; };  // (past the width: not used)
    auto put = [&](int slot, float4 v) { *follow_piece(st, slot, piece) = v; };
    auto meet = []() {  // LDS of one wave: what the lanes have stored is there for all of them
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
        __builtin_amdgcn_wave_barrier();
    };
    if (blockIdx.x < kFollowPairBlocks) {
        // lanes 2 i and 2 i + 1: the candidates of pair i; slots 0 .. 31 the rows, 32 + lane the centroids
        const uint32_t total = counts[1];
        for (uint64_t base = (blockIdx.x * 4 + wave) * 32; base < total; base += kFollowPairBlocks * 4 * 32) {
            const uint64_t e = base + (uint32_t)(lane >> 1);
            const uint2 ent = pairs[e < total ? e : base];
            const int64_t row = ent.x / (uint32_t)m;
            const int s = (int)(ent.x % (uint32_t)m), j = (int)((ent.y >> (8 * (lane & 1))) & 0xFFu);
            const float *xr[4], *cr[8];
#pragma unroll
            for (int u = 0; u < 4; ++u) {
                const uint32_t en = __shfl(ent.x, 2 * (8 * u + sub));
                xr[u] = a.x + (int64_t)(en / (uint32_t)m) * a.ld + (int64_t)(en % (uint32_t)m) * sd;
            }
#pragma unroll
            for (int u = 0; u < 8; ++u) cr[u] = a.cb + ((size_t)__shfl(s, 8 * u + sub) * k + __shfl(j, 8 * u + sub)) * sd;
            float4 px[4], pc[8];
            auto fetch = [&](int sl) {
#pragma unroll
                for (int u = 0; u < 4; ++u) px[u] = *reinterpret_cast<const float4 *>(xr[u] + at(sl));
#pragma unroll
                for (int u = 0; u < 8; ++u) pc[u] = *reinterpret_cast<const float4 *>(cr[u] + at(sl));
            };
            fetch(0);
            float acc = 0.0f;
            for (int sl = 0; sl < nsl; ++sl) {
                meet();  // the slice before has been read
#pragma unroll
                for (int u = 0; u < 4; ++u) put(8 * u + sub, px[u]);
#pragma unroll
                for (int u = 0; u < 8; ++u) put(32 + 8 * u + sub, pc[u]);
                meet();
                fetch(sl + 1 < nsl ? sl + 1 : sl);
                follow_slice<METRIC>(acc, st, lane >> 1, 32 + lane, sd - 32 * sl);
            }
            float d = METRIC == M_EUCLID ? sqrtf(acc) : acc;
            d = (d == d) ? d : inf;
            const float od = __shfl_xor(d, 1);
            const int oj = __shfl_xor(j, 1);
            if (e < total && (lane & 1) == 0) store_code<LBG>(a, row, s, (od < d || (od == d && oj < j)) ? oj : j);
        }
        return;
    }
    const uint32_t total = counts[0];
    if (total > kFollowMany) {  // uniform: a degenerate codebook or input; the codebook once per eight rows, all of it
        constexpr int room = 4 * kFollowSlots * 32;
        const unsigned block = blockIdx.x - kFollowPairBlocks;
        if (m == 1 && kRowsWg * sd + kRowsWgLdsFloats <= room) {
            wide_exact_rows_wg<METRIC, LBG>(a, sd, list, total, block, kFollowRowBlocks, stage[0]);
            return;
        }
        if (m > 1 && 4 * kWideRows * sd <= room) {
            wide_exact_groups<METRIC, LBG, true, true, kWideRows>(a, sd, list, total, stage[0] + wave * kWideRows * sd, lane, wave,
                                                                  block, kFollowRowBlocks);
            return;
        }
    }
    // one wave per row: slot 0 the row, slots 32 .. 95 up to 64 candidates at a time, in ascending order
    for (uint64_t e = (blockIdx.x - kFollowPairBlocks) * 4 + wave; e < total; e += kFollowRowBlocks * 4) {
        const uint32_t ent = list[e];
        const int64_t row = ent / (uint32_t)m;
        const int s = (int)(ent % (uint32_t)m);
        const float *xr = a.x + row * a.ld + (int64_t)s * sd;
        unsigned long long has[4];
        int nc = 0;
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const int j = 64 * q + lane;
            has[q] = __ballot(j < k && (e >= mask_cap || candidate_bit(masks + 2 * e, j)));
            nc += __popcll(has[q]);
        }
        float bd = inf;
        int bj = 0;
        for (int c0 = 0; c0 < nc; c0 += 64) {
            // candidate c0 + i -> its centroid
            auto centroid = [&](int i) {
                int left = c0 + i, j = 0;
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    const int here = __popcll(has[q]);
                    if (left >= 0 && left < here) {
                        unsigned long long w = has[q];
                        for (int u = left; u > 0; --u) w &= w - 1;
                        j = 64 * q + __ffsll(w) - 1;
                    }
                    left -= here;
                }
                return j;
            };
            const int live = nc - c0 < 64 ? nc - c0 : 64;
            const int j = lane < live ? centroid(lane) : 0;
            const int groups = (live + 7) / 8;  // uniform
            float4 px, pc[8];
            const float *cr[8];
#pragma unroll
            for (int u = 0; u < 8; ++u) cr[u] = a.cb + ((size_t)s * k + __shfl(j, 8 * u + sub)) * sd;
            auto fetch = [&](int sl) {
                px = *reinterpret_cast<const float4 *>(xr + at(sl));
#pragma unroll
                for (int u = 0; u < 8; ++u)
                    if (u < groups) pc[u] = *reinterpret_cast<const float4 *>(cr[u] + at(sl));
            };
            fetch(0);
            float acc = 0.0f;
            for (int sl = 0; sl < nsl; ++sl) {
                meet();
                if (lane < 8) put(0, px);
#pragma unroll
                for (int u = 0; u < 8; ++u)
                    if (u < groups) put(32 + 8 * u + sub, pc[u]);
                meet();
                fetch(sl + 1 < nsl ? sl + 1 : sl);
                follow_slice<METRIC>(acc, st, 0, 32 + (lane < live ? lane : 0), sd - 32 * sl);
            }
            const float raw = METRIC == M_EUCLID ? sqrtf(acc) : acc;
            const float d = lane < live && raw == raw ? raw : inf;  // a NaN distance never wins
            const uint32_t least = wave_umin(__float_as_uint(d));
            const int first = __ffsll(__ballot(__float_as_uint(d) == least)) - 1;  // ascending candidates: the lowest index
            const int fj = __builtin_amdgcn_readlane(j, first);
            const float fd = __uint_as_float(least);
            if (c0 == 0 || fd < bd) {
                bd = fd;
                bj = fj;
            }
            // ... unless it is centroid 0's, which is never displaced
            if (c0 == 0 && (has[0] & 1) && __builtin_amdgcn_readlane((int)(raw != raw), 0)) {
                bj = 0;
                break;
            }
        }
        if (lane == 0) store_code<LBG>(a, row, s, bj);
    }
}

}  // namespace vq

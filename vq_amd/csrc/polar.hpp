// The rotation update of OPQ, R = V U^T for A = U S V^T (src/opq.rs:180-183), without an SVD: R is the
// orthogonal polar factor of A^T, and for a non-singular A that factor is unique, so any convergent
// method gives the same matrix as the SVD does.  Newton-Schulz iteration on X_0 = A^T / s,
//     X_{k+1} = X_k (3 I - X_k^T X_k) / 2,
// converges to it when every singular value of X_0 lies in (0, sqrt 3): s = min(|A|_F, sqrt(|A|_1
// |A|_inf)) >= |A|_2 puts them in (0, 1].  A singular value sigma grows by 1.5 per step while it is
// small and converges quadratically once it is near 1: about log_1.5(cond) + 6 steps.  Scaled steps
// shorten the first phase: with every singular value in [l, 1], X (1.5 rho I - 0.5 rho^3 X^T X) with
// rho = sqrt(3 / (1 + l + l^2)) maps both ends of that interval to the same new lower bound
// l' = rho l (3 - rho^2 l^2) / 2 and everything between them into [l', 1] — small values grow by up to
// 2.6 per step.  l starts from a guess (1e-3 after the first, plain step); the map is valid for every
// singular value in (0, 1] whatever l is, so a wrong guess costs steps, never correctness.  The host
// passes rho_s with each step: the sequence that follows from the guess, then 1 (plain steps, which
// converge quadratically to the exact factor).  A matrix whose first error is below 0.005 is within
// 0.64 of orthogonal in the 2-norm (128 x the largest entry bounds it), so every singular value is
// above 0.6 already: it takes plain steps only — a scaled step would first spread them out.  A step is ONE launch (what a step costs is mostly the launch): a workgroup
// owns a strip of 16 columns (or a quarter of its result); its waves first make the strip of G = X^T X, one 16 x 16 tile each, in
// f64 on the matrix cores (v_mfma_f64_16x16x4_f64), leave M = 1.5 I - 0.5 G for the strip in LDS, meet,
// and then make their tiles of the strip of X M (the operands sit in L2; every operand of a tile is
// fetched before its first matrix instruction).  The first half also gives err_k = max |X_k^T X_k - I|;
// once it is below 1e-7 the update that follows squares it to rounding level and is the last one: the
// kernel of step s + 1 sees errs[s], returns at once and sets fin[s + 2], which the kernels after it
// read (the host has already enqueued them).  A matrix that has not
// converged within the step limit (singular or badly conditioned: cond above about 1e6) goes to the
// Jacobi SVD, which also completes the directions a singular A leaves open.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

namespace vq {

constexpr int kPolarMaxSteps = 56;
constexpr int kPolarMaxDim = 512;
constexpr double kPolarLastStepErr = 1e-7;
constexpr double kPolarPlainBelow = 0.005;  // no scaled steps at all when the first error is below this

typedef double polar_d4 __attribute__((ext_vector_type(4)));

// One 16 x 16 tile of a product over KS steps of four k: lane l supplies, per step,
// A[i = l % 16][k = 4 u + l / 16] and B[k = 4 u + l / 16][j = l % 16]; register v of lane l receives
// C[4 v + l / 16][l % 16].  Two chains of matrix instructions (even and odd steps), added at the end.
template <int KS> __device__ __forceinline__ polar_d4 polar_mfma(const double (&a)[KS], const double (&b)[KS]) {
    polar_d4 acc0 = {0.0, 0.0, 0.0, 0.0}, acc1 = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
    for (int u = 0; u < KS; u += 2) {
        acc0 = __builtin_amdgcn_mfma_f64_16x16x4f64(a[u], b[u], acc0, 0, 0, 0);
        acc1 = __builtin_amdgcn_mfma_f64_16x16x4f64(a[u + 1], b[u + 1], acc1, 0, 0, 0);
    }
    return acc0 + acc1;
}

// The same for any P (a multiple of 16), 16 steps' operands in flight at a time.  pa / pb point at the
// lane's first operands; they move on by sa / sb doubles per step.
__device__ __forceinline__ polar_d4 polar_tile(const double *__restrict__ pa, size_t sa,
                                               const double *__restrict__ pb, size_t sb, int P) {
    polar_d4 acc = {0.0, 0.0, 0.0, 0.0};
    for (int k0 = 0; k0 < P; k0 += 64) {
        double a[16], b[16];
#pragma unroll
        for (int u = 0; u < 16; ++u) {
            const bool in = k0 + 4 * u < P;
            const int kc = in ? k0 / 4 + u : P / 4 - 1;  // clamped: unconditional loads
            a[u] = pa[(size_t)kc * sa];
            b[u] = in ? pb[(size_t)kc * sb] : 0.0;
            a[u] = in ? a[u] : 0.0;
        }
        acc = acc + polar_mfma<16>(a, b);
    }
    return acc;
}

// Step s: Xout = Xin (1.5 r I - 0.5 r^3 Xin^T Xin) with r = rho when the error of step 0 was at
// least kPolarPlainBelow, else 1; errs[s] = max |Xin^T Xin - I| over the dim x dim block that holds
// data (NaN counts as infinite).  P x P matrices, row-major, zero beyond dim.  Grid: four workgroups per
// column strip (P / 16 strips, of min(P / 16, 8) waves): a strip's products on one compute unit are bound by
// its matrix instructions (64 cycles each, 4 us of a step at P = 128), so each of the four makes all of M and a
// quarter of the tiles of the result.  P = 128: 13.2 us per step with one workgroup per strip, 7.7 with four.
// Dynamic LDS: P * 16 doubles.
// PT = 8: P = 128, every operand of a tile fetched at once, and the rows of Xin for the second half already
// on their way during the first; 0: any P.
template <int PT>
static __global__ void __launch_bounds__(512) k_polar_step(const double *__restrict__ Xin, int P, int dim, int s,
                                                           double rho, unsigned long long *__restrict__ errs,
                                                           int *__restrict__ fin, double *__restrict__ Xout) {
    extern __shared__ __attribute__((aligned(16))) double m_strip[];  // M[c][16 tj + jj] at [c * 16 + jj]
    const double prev = s > 0 ? __longlong_as_double((long long)errs[s - 1]) : 2.0;
    const bool dead = fin[s] != 0 || prev < kPolarLastStepErr;
    if (dead) {  // the same in every workgroup
        if (blockIdx.x == 0 && threadIdx.x == 0) fin[s + 1] = 1;
        return;
    }
    const double first = s > 0 ? __longlong_as_double((long long)errs[0]) : 0.0;
    const double r = first >= kPolarPlainBelow ? rho : 1.0;
    const double ca = 1.5 * r, cb = 0.5 * r * r * r;
    const int nt = P / 16, tj = (int)blockIdx.x % nt, share = (int)blockIdx.x / nt;
    const int lane = threadIdx.x & 63, kk = lane >> 4, jj = lane & 15;
    const int w = threadIdx.x >> 6, nw = blockDim.x >> 6;
    double e = 0.0;
    auto emit = [&](const polar_d4 &acc, int ti) {
#pragma unroll
        for (int v = 0; v < 4; ++v) {
            const int i = 16 * ti + 4 * v + kk, j = 16 * tj + jj;
            const double d = i == j ? 1.0 : 0.0, g = acc[v];
            m_strip[i * 16 + jj] = ca * d - cb * g;
            if (i < dim && j < dim) {
                const double dev = fabs(g - d);
                e = (dev <= e) ? e : (dev == dev ? dev : __builtin_inf());
            }
        }
    };
    auto report = [&]() {  // by one of a strip's workgroups
        if (share) return;
#pragma unroll
        for (int off = 32; off > 0; off >>= 1) {
            const double o = __shfl_xor(e, off);
            e = o > e ? o : e;
        }
        // non-negative doubles order like their bit patterns
        if (lane == 0) atomicMax(errs + s, (unsigned long long)__double_as_longlong(e));
    };
    if constexpr (PT > 0) {
        static_assert(PT == 8, "eight waves, a tile each");
        constexpr int KS = 4 * PT, PP = 16 * PT;
        const int ti = w;  // one tile per wave
        // G[i][j] = sum_r X[r][i] X[r][j]: both operands run down a column of X, four rows per step
        double a[KS], b[KS];
        const double *pa = Xin + (size_t)kk * PP + 16 * ti + jj, *pb = Xin + (size_t)kk * PP + 16 * tj + jj;
#pragma unroll
        for (int u = 0; u < KS; ++u) {
            a[u] = pa[(size_t)u * 4 * PP];
            b[u] = pb[(size_t)u * 4 * PP];
        }
        // the second half's rows of Xin: Xout[r][j] = sum_c Xin[r][c] M[c][j], A runs along a row.  Two of
        // the strip's tiles per workgroup, four waves a tile with a quarter of the sum each; a lane has two
        // consecutive c of every eight (16-byte loads)
        const int to = 2 * share + (w >> 2), c0 = (w & 3) * (PP / 4) + 2 * kk;
        const double2 *pr = reinterpret_cast<const double2 *>(Xin + (size_t)(16 * to + jj) * PP + c0);
        double2 r2[KS / 8];
#pragma unroll
        for (int v = 0; v < KS / 8; ++v) r2[v] = pr[4 * v];
        emit(polar_mfma<KS>(a, b), ti);
        report();
        __syncthreads();
        double a2[KS / 4], b2[KS / 4];
#pragma unroll
        for (int v = 0; v < KS / 8; ++v) {
            a2[2 * v] = r2[v].x;
            a2[2 * v + 1] = r2[v].y;
            b2[2 * v] = m_strip[(c0 + 8 * v) * 16 + jj];
            b2[2 * v + 1] = m_strip[(c0 + 8 * v + 1) * 16 + jj];
        }
        const polar_d4 acc = polar_mfma<KS / 4>(a2, b2);
        __syncthreads();  // the strip becomes the quarters' sums, [wave][v][lane]
#pragma unroll
        for (int v = 0; v < 4; ++v) m_strip[(w * 4 + v) * 64 + lane] = acc[v];
        __syncthreads();
        const double *q = m_strip + (w & 4) * 256 + (w & 3) * 64 + lane;  // this thread: v = w % 4 of its tile
        Xout[(size_t)(16 * to + 4 * (w & 3) + kk) * PP + 16 * tj + jj] = (q[0] + q[256]) + (q[512] + q[768]);
    } else {
        for (int ti = w; ti < nt; ti += nw)
            emit(polar_tile(Xin + (size_t)kk * P + 16 * ti + jj, 4 * (size_t)P, Xin + (size_t)kk * P + 16 * tj + jj,
                            4 * (size_t)P, P),
                 ti);
        report();
        __syncthreads();
        for (int ti = 4 * w + share; ti < nt; ti += 4 * nw) {
            const polar_d4 acc = polar_tile(Xin + (size_t)(16 * ti + jj) * P + kk, 4, m_strip + kk * 16 + jj, 64, P);
#pragma unroll
            for (int v = 0; v < 4; ++v) Xout[(size_t)(16 * ti + 4 * v + kk) * P + 16 * tj + jj] = acc[v];
        }
    }
}

// ---- the start and the end of the iteration on the device ------------------------------------------
// A stays where the cross-covariance left it; the elements are rounded to f32 first (the reference's A is
// a matrix of f32).  On the host the two norms, the transposed copy and the way there and back took 220 us of
// a rotation update at 128 dimensions, the steps themselves 190.

// The step tables of one iteration.
struct PolarTables {
    unsigned long long *errs;  // [kPolarMaxSteps]
    int *fin;                  // [kPolarMaxSteps + 2]
    int *bad;                  // A is zero or not finite: the steps return at once
};

__device__ __forceinline__ double polar_in(const double *A, size_t e) { return (double)(float)A[e]; }

// Workgroup b: of rows 16 b .. 16 b + 15, the sums of |a| by column (col_part[b][dim]) and by row, and the
// rows' sums of squares.  256 threads.
static __global__ void __launch_bounds__(256) k_polar_norms(const double *__restrict__ A, int dim,
                                                            double *__restrict__ col_part, double *__restrict__ row_sum,
                                                            double *__restrict__ row_sq) {
    const int i0 = 16 * blockIdx.x, rows = dim - i0 < 16 ? dim - i0 : 16;
    for (int j = threadIdx.x; j < dim; j += 256) {
        double v[16], c = 0.0;
#pragma unroll
        for (int u = 0; u < 16; ++u) v[u] = polar_in(A, (size_t)(i0 + (u < rows ? u : 0)) * dim + j);
#pragma unroll
        for (int u = 0; u < 16; ++u) c += u < rows ? fabs(v[u]) : 0.0;
        col_part[(size_t)blockIdx.x * dim + j] = c;
    }
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    for (int u = wave; u < rows; u += 4) {
        double a = 0.0, q = 0.0;
        for (int j = lane; j < dim; j += 64) {
            const double v = polar_in(A, (size_t)(i0 + u) * dim + j);
            a += fabs(v);
            q += v * v;
        }
#pragma unroll
        for (int off = 32; off > 0; off >>= 1) {
            a += __shfl_xor(a, off);
            q += __shfl_xor(q, off);
        }
        if (lane == 0) {
            row_sum[i0 + u] = a;
            row_sq[i0 + u] = q;
        }
    }
}

// X = A^T / scale, P x P, zero beyond dim, and cleared tables.  P / 16 workgroups of 256 threads, each with
// its own copy of the scale.
static __global__ void __launch_bounds__(256) k_polar_start(const double *__restrict__ A, int dim, int P,
                                                            const double *__restrict__ col_part,
                                                            const double *__restrict__ row_sum,
                                                            const double *__restrict__ row_sq, PolarTables tb,
                                                            double *__restrict__ X) {
    __shared__ double red[3][4];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, strips = (dim + 15) / 16;
    double n1 = 0.0, ni = 0.0, fro = 0.0;
    for (int j = tid; j < dim; j += 256) {
        double c = 0.0;
        for (int b = 0; b < strips; ++b) c += col_part[(size_t)b * dim + j];
        n1 = fmax(n1, c);
        ni = fmax(ni, row_sum[j]);
        fro += row_sq[j];  // (a NaN stays in this one)
    }
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) {
        n1 = fmax(n1, __shfl_xor(n1, off));
        ni = fmax(ni, __shfl_xor(ni, off));
        fro += __shfl_xor(fro, off);
    }
    if (lane == 0) {
        red[0][wave] = n1;
        red[1][wave] = ni;
        red[2][wave] = fro;
    }
    __syncthreads();
    n1 = fmax(fmax(red[0][0], red[0][1]), fmax(red[0][2], red[0][3]));
    ni = fmax(fmax(red[1][0], red[1][1]), fmax(red[1][2], red[1][3]));
    fro = (red[2][0] + red[2][1]) + (red[2][2] + red[2][3]);
    // two upper bounds of the largest singular value; the smaller one
    const double by_sums = sqrt(n1) * sqrt(ni), by_squares = sqrt(fro);
    const double scale = by_sums < by_squares ? by_sums : by_squares;
    const bool ok = scale > 0.0 && scale < __builtin_inf();
    if (blockIdx.x == 0) {
        if (tid < kPolarMaxSteps) tb.errs[tid] = 0ull;
        if (tid < kPolarMaxSteps + 2) tb.fin[tid] = tid == 0 && !ok ? 1 : 0;
        if (tid == 0) tb.bad[0] = ok ? 0 : 1;
    }
    const double inv = ok ? 1.0 / scale : 0.0;
    const int i0 = 16 * blockIdx.x;
    for (int j = tid; j < P; j += 256) {
        double v[16];
#pragma unroll
        for (int u = 0; u < 16; ++u) {
            const bool in = i0 + u < dim && j < dim;
            v[u] = polar_in(A, in ? (size_t)(i0 + u) * dim + j : 0);
            v[u] = in && ok ? v[u] * inv : 0.0;
        }
#pragma unroll
        for (int u = 0; u < 16; ++u) X[(size_t)j * P + i0 + u] = v[u];
    }
}

// After `steps` steps: R = the iterate behind the first step whose error was below kPolarLastStepErr, in
// f32, and status 1; 0 where there is none yet, -1 where the iteration could not begin.
static __global__ void __launch_bounds__(256) k_polar_finish(const double *__restrict__ X0, const double *__restrict__ X1,
                                                             int P, int dim, PolarTables tb, int steps,
                                                             float *__restrict__ R, int *status) {
    int last = -1;
    for (int t = steps - 1; t >= 0; --t)
        if (__longlong_as_double((long long)tb.errs[t]) < kPolarLastStepErr) last = t;
    const bool bad = tb.bad[0] != 0;
    if (blockIdx.x == 0 && threadIdx.x == 0) *status = bad ? -1 : (last >= 0 ? 1 : 0);
    if (bad || last < 0) return;
    const double *X = (last + 1) & 1 ? X1 : X0;
    for (int e = blockIdx.x * 256 + threadIdx.x; e < dim * dim; e += gridDim.x * 256)
        R[e] = (float)X[(size_t)(e / dim) * P + e % dim];
}

}  // namespace vq

// libvqhip — entry points around the assignment for ResidualQuantizer and
// OptimizedProductQuantizer (declared in include/vq_hip.h).
#include <hip/hip_runtime.h>
#include <hip/hip_fp16.h>

#include <algorithm>
#include <cmath>
#include <cstring>
#include <vector>

#include "ctx.hpp"
#include "rvq_opq.hpp"
#include "resident_rules.hpp"
#include "procrustes_host.hpp"
#include "polar.hpp"

using namespace vqh;

namespace {

template <typename CodeT>
int32_t residual_sub(vq_ctx *ctx, float *d_res, int64_t n, int64_t ld, int32_t dim, int32_t k, int32_t k_max,
                     const float *d_codebook, const CodeT *d_codes) {
    if (!ctx) return VQ_ERR_INVALID_ARG;
    if (n == 0) return VQ_OK;
    if (!d_res || !d_codebook || !d_codes || n < 0 || dim <= 0 || ld < dim || k <= 0 || k > k_max)
        return fail(ctx, VQ_ERR_INVALID_ARG, "Invalid parameter");
    VQ_HIP(ctx, hipSetDevice(ctx->device));
    if (dim % 4 == 0 && ld % 4 == 0 &&
        ((reinterpret_cast<uintptr_t>(d_res) | reinterpret_cast<uintptr_t>(d_codebook)) & 15) == 0)
        hipLaunchKernelGGL(vq::k_residual_sub4<CodeT>, dim3(cdiv(n * (dim / 4), 1024)), dim3(256), 0, ctx->stream,
                           d_res, n, ld, dim / 4, d_codebook, d_codes, (const uint8_t *)nullptr, (CodeT *)nullptr, 0, 0,
                           (uint8_t *)nullptr, (const float *)d_res, ld);
    else
        hipLaunchKernelGGL(vq::k_residual_sub<CodeT>, dim3(cdiv(n * dim, 256)), dim3(256), 0, ctx->stream, d_res, n,
                           ld, dim, d_codebook, d_codes, 1);
    VQ_HIP(ctx, hipGetLastError());
    return VQ_OK;
}

inline int32_t assign_any(vq_ctx *ctx, int32_t metric, const float *x, int64_t n, int64_t ld, int32_t dim,
                          int32_t k, const float *cb, uint8_t *codes) {
    return assign_codes(ctx, metric, x, n, ld, 1, dim, k, cb, codes);
}
inline int32_t assign_any(vq_ctx *ctx, int32_t metric, const float *x, int64_t n, int64_t ld, int32_t dim,
                          int32_t k, const float *cb, uint16_t *codes) {
    return assign_codes_u16(ctx, metric, x, n, ld, 1, dim, k, cb, codes);
}

template <typename CodeT>
int32_t rvq_encode(vq_ctx *ctx, int32_t metric, const float *d_x, int64_t n, int64_t ld, int32_t dim, int32_t stages,
                   int32_t k, int32_t k_max, const float *d_codebooks, float epsilon, CodeT *d_codes,
                   uint8_t *d_stages_used, uint16_t *d_recon_f16) {
    if (!ctx) return VQ_ERR_INVALID_ARG;
    if (n == 0) return VQ_OK;
    if (!d_x || !d_codebooks || !d_codes || n < 0 || dim <= 0 || ld < dim || stages < 0 || k <= 0 || k > k_max ||
        stages > 255)
        return fail(ctx, VQ_ERR_INVALID_ARG, "Invalid parameter");
    VQ_HIP(ctx, hipSetDevice(ctx->device));
    hipStream_t st = ctx->stream;
    if (stages > 0 && assign_few_applicable(ctx, n, 1, dim)) {
        const size_t lds = sizeof(float) * 2 * ((size_t)dim + 3);
#define FEW(M)                                                                                                      \
    hipLaunchKernelGGL((vq::k_rvq_few<M, CodeT>), dim3((unsigned)n), dim3(256), lds, st, d_x, ld, dim, stages, k,      \
                       d_codebooks, epsilon, d_codes, d_stages_used, d_recon_f16)
        switch (metric) {
        case VQ_SQEUCLIDEAN: FEW(vq::M_SQ); break;
        case VQ_EUCLIDEAN: FEW(vq::M_EUCLID); break;
        case VQ_COSINE: FEW(vq::M_COS); break;
        case VQ_MANHATTAN: FEW(vq::M_L1); break;
        default: return fail(ctx, VQ_ERR_UNSUPPORTED, "metric %d has no kernel", metric);
        }
#undef FEW
        VQ_HIP(ctx, hipGetLastError());
        return VQ_OK;
    }
    // Widths that every stage's assignment would pad: rows and codebooks once, the copy of the rows is the residual
    // (137,227 x 100, five stages, k = 16 412 -> 297 us, 1M x 100, eight stages, k = 256 4.60 -> 2.58 ms)
    const float *rx = d_x, *rcb = d_codebooks;
    int64_t rld = ld;
    int w = dim;
    const int wp = stages > 1 && k >= 2 ? encode_pad_width(ctx, metric, d_x, n, ld, 1, dim, std::min(k, 256), d_codebooks) : 0;
    const size_t pad_bytes = sizeof(float) * ((size_t)n + (size_t)stages * k) * wp;
    const bool padded = wp > dim && pad_bytes <= kPadKeep && ensure(ctx, ctx->pad_rows, pad_bytes) == VQ_OK;
    if (padded) {
        float *px = (float *)ctx->pad_rows.p, *pcb = px + (size_t)n * wp;
        pad_blocks(ctx, d_x, n, ld, 1, dim, wp, px);
        pad_blocks(ctx, d_codebooks, (int64_t)stages * k, dim, 1, dim, wp, pcb);
        rx = px, rcb = pcb, rld = wp, w = wp;
    }
    const bool vec4 = w % 4 == 0 && (reinterpret_cast<uintptr_t>(rcb) & 15) == 0;
    // The first stage reads the caller's rows where they lie and writes the first residual; the last
    // stage leaves the residual alone.  One stage then needs no residual buffer at all.
    const bool direct = !padded && vec4 && rld % 4 == 0 && (reinterpret_cast<uintptr_t>(rx) & 15) == 0;
    const bool need_res = !padded && (stages > 1 || (stages == 1 && !direct));
    if (need_res) VQ_TRY(ensure(ctx, ctx->tmp_c, sizeof(float) * (size_t)n * w));   // residual
    const size_t codes_bytes = ((size_t)n * sizeof(CodeT) + 3) & ~(size_t)3;
    VQ_TRY(ensure(ctx, ctx->tmp_e, 2 * codes_bytes + 2 * (size_t)n + 16));  // stage codes (two), active, used
    VQ_TRY(ensure(ctx, ctx->tmp_a, sizeof(float) * (size_t)n));         // row norms
    float *norms = (float *)ctx->tmp_a.p;
    float *res = padded ? (float *)ctx->pad_rows.p : (float *)ctx->tmp_c.p;
    CodeT *stage_codes[2] = {(CodeT *)ctx->tmp_e.p, (CodeT *)((uint8_t *)ctx->tmp_e.p + codes_bytes)};
    uint8_t *active = (uint8_t *)ctx->tmp_e.p + 2 * codes_bytes;
    uint8_t *used = d_stages_used ? d_stages_used : active + n;
    // With no norm test between the stages (epsilon <= 0: every row uses every stage) the update of
    // the residual by a stage's centroids waits for the next stage's assignment, where that pass can
    // take it along: one pass over the rows per stage instead of two.
    bool defer = false;
    if constexpr (sizeof(CodeT) == 1)
        defer = !(epsilon > 0.0f) && stages > 1 && k >= 2 && vec4 &&
                assign_pending_fusable(ctx, metric, res, n, w, w, k, rcb);
    if (need_res && !direct)
        VQ_HIP(ctx, hipMemcpy2DAsync(res, sizeof(float) * w, rx, sizeof(float) * rld, sizeof(float) * w,
                                     (size_t)n, hipMemcpyDeviceToDevice, st));
    hipLaunchKernelGGL(vq::k_rvq_begin, dim3(cdiv(n, 256)), dim3(256), 0, st, active, used, n);
    // the tables of all stages in one launch, as far as they are small beside the rows
    struct Stages {
        vq_ctx::StageTables &t;
        ~Stages() { t = vq_ctx::StageTables(); }
    } tables{ctx->stage_tables};
    if (sizeof(CodeT) == 1 && stages > 1 && (int64_t)stages * k <= n) {
        tables.t.cb = rcb;
        tables.t.stages = stages;
    }
    const float *pend_cb = nullptr;  // the stage whose update of the residual is still to come
    const CodeT *pend_codes = nullptr;
    bool pend_from_x = false;        // ... and reads the caller's rows
    for (int s = 0; s < stages; ++s) {
        const float *cb = rcb + (size_t)s * k * w;
        tables.t.stage = s;
        CodeT *cur = stage_codes[s & 1];
        const bool from_x = direct && s == 0;
        const float *rows = from_x ? rx : res;
        const int64_t rows_ld = from_x ? rld : (int64_t)w;
        if (k < 2) {  // src/rvq.rs:186-187
            hipLaunchKernelGGL(vq::k_fill<CodeT>, dim3(cdiv(n, 256)), dim3(256), 0, st, cur, n, (CodeT)0);
        } else if (pend_cb) {
            if constexpr (sizeof(CodeT) == 1) {
                const PendingUpdate pu{pend_cb, pend_codes, pend_from_x ? rx : nullptr, pend_from_x ? rld : 0};
                VQ_TRY(assign_codes(ctx, metric, res, n, w, 1, w, k, cb, cur, nullptr, nullptr, &pu));
            }
            pend_cb = nullptr;
        } else {
            VQ_TRY(assign_any(ctx, metric, rows, n, rows_ld, w, k, cb, cur));
        }
        if (s == stages - 1 || defer) {
            hipLaunchKernelGGL(vq::k_rvq_stage_record<CodeT>, dim3(cdiv(n, 256)), dim3(256), 0, st, n,
                               (const CodeT *)cur, (const uint8_t *)active, d_codes, stages, s, used);
            if (s == stages - 1) break;
            pend_cb = cb;
            pend_codes = cur;
            pend_from_x = from_x;
            continue;
        }
        if (vec4 && epsilon > 0.0f) {
            hipLaunchKernelGGL(vq::k_rvq_stage_step4<CodeT>, dim3(cdiv(n, 64)), dim3(64), 0, st, res, n, w, cb,
                               (const CodeT *)cur, d_codes, stages, s, active, used, rows, rows_ld, epsilon);
            continue;
        }
        if (vec4)
            hipLaunchKernelGGL(vq::k_residual_sub4<CodeT>, dim3(cdiv(n * (w / 4), 1024)), dim3(256), 0, st, res, n,
                               (int64_t)w, w / 4, cb, (const CodeT *)cur, (const uint8_t *)active, d_codes,
                               stages, s, used, rows, rows_ld);
        else
            hipLaunchKernelGGL(vq::k_rvq_stage_apply<CodeT>, dim3(cdiv(n * w, 256)), dim3(256), 0, st, res, n, w,
                               cb, (const CodeT *)cur, d_codes, stages, s, (const uint8_t *)active, used);
        if (epsilon > 0.0f) {  // a norm is never below a non-positive threshold
            hipLaunchKernelGGL(vq::k_row_norms, dim3(cdiv(n, 64)), dim3(64), 0, st, res, n, (int64_t)w, w,
                               norms);
            hipLaunchKernelGGL(vq::k_rvq_stage_stop, dim3(cdiv(n, 256)), dim3(256), 0, st, norms, n, epsilon,
                               active);
        }
    }
    if (d_recon_f16) {
        const bool vec4 = dim % 4 == 0 && (reinterpret_cast<uintptr_t>(d_codebooks) & 15) == 0;
        const int cols = vq::rvq_recon_columns(n, stages, k, dim);
        if (vec4 && cols && n * dim >= (1 << 21) && (reinterpret_cast<uintptr_t>(d_recon_f16) & 15) == 0) {
            const size_t lds = sizeof(float) * (size_t)stages * k * cols;
            auto kern = vq::k_rvq_recon_resident<CodeT>;
            VQ_HIP(ctx, hipFuncSetAttribute(reinterpret_cast<const void *>(kern),
                                            hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
            // (up to 32 groups: a multiple of eight workgroups each, see the kernel)
            const unsigned groups = cdiv(dim, cols), wgs = groups <= 32 ? 256u / groups / 8 * 8 : std::max(1u, 256u / groups);
            hipLaunchKernelGGL(kern, dim3(wgs, groups), dim3(1024), lds, st, n, dim, k, cols, d_codebooks,
                               (const CodeT *)d_codes, stages, (const uint8_t *)used, (vq::rot_u32x4 *)d_recon_f16);
        } else if (vec4 && (reinterpret_cast<uintptr_t>(d_recon_f16) & 7) == 0)
            hipLaunchKernelGGL(vq::k_rvq_recon4_f16<CodeT>, dim3(cdiv(n * (dim / 4), 1024)), dim3(256), 0, st, n,
                               dim / 4, k, d_codebooks, (const CodeT *)d_codes, stages, (const uint8_t *)used,
                               d_recon_f16);
        else
            hipLaunchKernelGGL(vq::k_rvq_recon_f16<CodeT>, dim3(cdiv(n * dim, 256)), dim3(256), 0, st, n, dim, k,
                               d_codebooks, (const CodeT *)d_codes, stages, (const uint8_t *)used, d_recon_f16);
    }
    VQ_HIP(ctx, hipGetLastError());
    return VQ_OK;
}

}  // namespace

namespace {

// Enqueues the steps from .. upto - 1 of the iteration in X[0], X[1] (polar.hpp).  low: the assumed lower
// bound of the singular values, 1e-3 before step 0.
int32_t polar_steps(vq_ctx *ctx, double *const (&X)[2], int dim, int from, int upto, double &low, unsigned long long *errs,
                    int *fin) {
    const int P = (dim + 15) / 16 * 16;
    const unsigned strips = (unsigned)(P / 16), waves = strips < 8u ? strips : 8u;
    const size_t lds = sizeof(double) * 16 * (size_t)P;
    if (lds > 48 * 1024)
        VQ_HIP(ctx, hipFuncSetAttribute(reinterpret_cast<const void *>(vq::k_polar_step<0>),
                                        hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
    for (int s = from; s < upto; ++s) {
        double rho = 1.0;
        if (s > 0 && low < 0.9) {
            rho = std::sqrt(3.0 / (1.0 + low + low * low));
            low = rho * low * (3.0 - rho * rho * low * low) * 0.5;
        }
        hipLaunchKernelGGL((P == 128 ? vq::k_polar_step<8> : vq::k_polar_step<0>), dim3(4 * strips), dim3(64 * waves), lds,
                           ctx->stream, (const double *)X[s & 1], P, dim, s, rho, errs, fin, X[(s + 1) & 1]);
    }
    VQ_HIP(ctx, hipGetLastError());
    return VQ_OK;
}

// R = the orthogonal polar factor of A^T by Newton-Schulz steps (polar.hpp).  *done = false when the
// iteration has not converged within its step limit (the caller then takes the SVD).
int32_t polar_newton_schulz(vq_ctx *ctx, const double *h_A, int dim, double *h_R, bool *done) {
    *done = false;
    if (dim > vq::kPolarMaxDim) return VQ_OK;
    const int P = (dim + 15) / 16 * 16;
    const size_t total = (size_t)P * P;
    // |A|_1 and |A|_inf: largest column and row sums of |a|
    std::vector<double> colsum((size_t)dim, 0.0);
    double norm_inf = 0.0;
    for (int i = 0; i < dim; ++i) {
        double r = 0.0;
        for (int j = 0; j < dim; ++j) {
            const double v = std::fabs(h_A[(size_t)i * dim + j]);
            r += v;
            colsum[j] += v;
        }
        norm_inf = std::max(norm_inf, r);
    }
    double norm_1 = 0.0;
    for (double c : colsum) norm_1 = std::max(norm_1, c);
    double fro = 0.0;
    for (size_t e = 0; e < (size_t)dim * dim; ++e) fro += h_A[e] * h_A[e];
    // two upper bounds of the largest singular value; the smaller one
    const double scale = std::min(std::sqrt(fro), std::sqrt(norm_1) * std::sqrt(norm_inf));
    if (!(scale > 0.0) || !std::isfinite(scale)) return VQ_OK;  // zero or non-finite: the SVD path decides
    std::vector<double> x0(total, 0.0);  // A^T / scale, zero-padded to P x P
    const double inv = 1.0 / scale;
    for (int i = 0; i < dim; ++i)
        for (int j = 0; j < dim; ++j) x0[(size_t)j * P + i] = h_A[(size_t)i * dim + j] * inv;
    VQ_TRY(ensure(ctx, ctx->tmp_a, sizeof(double) * total));
    VQ_TRY(ensure(ctx, ctx->tmp_b, sizeof(double) * total));
    VQ_TRY(ensure(ctx, ctx->tmp_f, 1024));
    double *X[2] = {(double *)ctx->tmp_a.p, (double *)ctx->tmp_b.p};
    unsigned long long *errs = (unsigned long long *)ctx->tmp_f.p;  // kPolarMaxSteps of them, then the flags
    int *fin = (int *)(errs + vq::kPolarMaxSteps);
    static_assert(sizeof(unsigned long long) * vq::kPolarMaxSteps + sizeof(int) * (vq::kPolarMaxSteps + 2) <= 1024,
                  "step tables");
    hipStream_t st = ctx->stream;
    VQ_HIP(ctx, hipMemsetAsync(ctx->tmp_f.p, 0, 1024, st));
    VQ_HIP(ctx, hipMemcpyAsync(X[0], x0.data(), sizeof(double) * total, hipMemcpyHostToDevice, st));
    unsigned long long h_errs[vq::kPolarMaxSteps];
    int s = 0, last = -1;
    double low = 1e-3;
    while (s < vq::kPolarMaxSteps && last < 0) {
        const int upto = std::min(vq::kPolarMaxSteps, s == 0 ? 16 : s + 6);
        VQ_TRY(polar_steps(ctx, X, dim, s, upto, low, errs, fin));
        s = upto;
        VQ_HIP(ctx, hipMemcpyAsync(h_errs, errs, sizeof(unsigned long long) * s, hipMemcpyDeviceToHost, st));
        VQ_HIP(ctx, hipStreamSynchronize(st));
        for (int t = 0; t < s && last < 0; ++t) {
            double e;
            std::memcpy(&e, &h_errs[t], sizeof e);
            if (e < vq::kPolarLastStepErr) last = t;
        }
    }
    if (last < 0) return VQ_OK;
    std::vector<double> r(total);
    VQ_HIP(ctx, hipMemcpyAsync(r.data(), X[(last + 1) & 1], sizeof(double) * total, hipMemcpyDeviceToHost, st));
    VQ_HIP(ctx, hipStreamSynchronize(st));
    for (int i = 0; i < dim; ++i)
        for (int j = 0; j < dim; ++j) h_R[(size_t)i * dim + j] = r[(size_t)i * P + j];
    *done = true;
    return VQ_OK;
}

// R = V U^T of the one-sided Jacobi SVD: on the device for even dim up to kJacobiMax, else on the host.
int32_t procrustes_svd(vq_ctx *ctx, const double *h_A, int dim, double *h_R) {
    if (dim > vq::kJacobiMax || dim % 2 != 0) {
        vqh::procrustes_host(h_A, (size_t)dim, h_R);
        return VQ_OK;
    }
    const size_t total = (size_t)dim * dim;
    const int half = dim / 2;
    VQ_TRY(ensure(ctx, ctx->tmp_a, sizeof(double) * total));
    VQ_TRY(ensure(ctx, ctx->tmp_b, sizeof(double) * total));
    VQ_TRY(ensure(ctx, ctx->tmp_c, sizeof(double) * (total + dim)));
    VQ_TRY(ensure(ctx, ctx->tmp_d, sizeof(double) * total));
    VQ_TRY(ensure(ctx, ctx->tmp_e, sizeof(double2) * (size_t)vq::kJacobiSweeps * (dim - 1) * half));
    VQ_TRY(ensure(ctx, ctx->tmp_f, 256));
    double *d_A = (double *)ctx->tmp_a.p, *d_vt = (double *)ctx->tmp_b.p, *d_uhat = (double *)ctx->tmp_c.p;
    double *d_sv = d_uhat + total;
    double *d_out = (double *)ctx->tmp_d.p;
    double2 *d_rot = (double2 *)ctx->tmp_e.p;
    int *d_rounds = (int *)ctx->tmp_f.p;
    VQ_HIP(ctx, hipMemcpyAsync(d_A, h_A, sizeof(double) * total, hipMemcpyHostToDevice, ctx->stream));
    constexpr int kLanes = 8;
    const size_t lds = sizeof(double) * (size_t)dim * vq::kJacobiStride;
    VQ_HIP(ctx, hipFuncSetAttribute(reinterpret_cast<const void *>(vq::k_jacobi_sweeps<kLanes>),
                                    hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
    hipLaunchKernelGGL(vq::k_jacobi_sweeps<kLanes>, dim3(1), dim3(64 * kLanes), lds, ctx->stream, (const double *)d_A,
                       dim, d_rot, d_rounds, d_uhat, d_sv);
    hipLaunchKernelGGL(vq::k_jacobi_accumulate, dim3(dim), dim3(64), 0, ctx->stream, (const double2 *)d_rot,
                       (const int *)d_rounds, dim, d_vt);
    hipLaunchKernelGGL(vq::k_jacobi_product, dim3((unsigned)cdiv(total, 256)), dim3(256), 0, ctx->stream,
                       (const double *)d_vt, (const double *)d_uhat, dim, d_out);
    VQ_HIP(ctx, hipGetLastError());
    std::vector<double> sv((size_t)dim);
    VQ_HIP(ctx, hipMemcpyAsync(h_R, d_out, sizeof(double) * total, hipMemcpyDeviceToHost, ctx->stream));
    VQ_HIP(ctx, hipMemcpyAsync(sv.data(), d_sv, sizeof(double) * dim, hipMemcpyDeviceToHost, ctx->stream));
    VQ_HIP(ctx, hipStreamSynchronize(ctx->stream));
    // A singular A leaves directions of U open (their columns came back as zero or as rounding
    // noise): complete them on the host and form the product again.  Rare; a full-rank A ends here.
    double top = 0.0;
    for (double v : sv) top = std::max(top, v);
    bool open = false;
    for (double v : sv) open = open || !(top > 0.0 && v > vqh::kNullRel * top);
    if (open) {
        std::vector<double> Ut(total), Vt(total);
        VQ_HIP(ctx, hipMemcpyAsync(Ut.data(), d_uhat, sizeof(double) * total, hipMemcpyDeviceToHost, ctx->stream));
        VQ_HIP(ctx, hipMemcpyAsync(Vt.data(), d_vt, sizeof(double) * total, hipMemcpyDeviceToHost, ctx->stream));
        VQ_HIP(ctx, hipStreamSynchronize(ctx->stream));
        vqh::complete_null_columns(Ut, Vt, sv, (size_t)dim);
        vqh::product_v_ut(Vt, Ut, (size_t)dim, h_R);
    }
    return VQ_OK;
}

// d_y^T d_x to tmp_b, dim x dim in f64.
int32_t cross_cov_device(vq_ctx *ctx, const float *d_y, const float *d_x, int64_t n, int32_t dim) {
    // chunks of 2048 rows up to dim 128; longer chunks for larger matrices, so that the partial
    // sums (one dim x dim matrix per chunk) stay at about 64 B per row
    const int64_t scale = ((int64_t)dim + 127) / 128;
    // and shorter ones where that would leave fewer than 256 workgroups (a chunk has scale^2): 50,000 x 128
    // was 25 workgroups and 265 us, now 34 us
    const int64_t rows_per_chunk =
        std::min<int64_t>(2048, std::max<int64_t>(128, (n / 256 + 3) / 4 * 4)) * scale * scale;
    const int chunks = (int)cdiv(n, rows_per_chunk);
    const int total = dim * dim;
    VQ_TRY(ensure(ctx, ctx->tmp_a, sizeof(double) * (size_t)chunks * total));
    VQ_TRY(ensure(ctx, ctx->tmp_b, sizeof(double) * (size_t)total));
    VQ_TRY(ensure(ctx, ctx->tmp_c, sizeof(double) * (size_t)total * ((chunks + 31) / 32)));
    if (dim >= 16) {
        const int nt_all = (int)cdiv(dim, 16), full = nt_all / 8, rest = nt_all % 8;
        double *part = (double *)ctx->tmp_a.p;
#define CROSSCOV(NT, B0, Z)                                                                                 \
    hipLaunchKernelGGL((vq::k_crosscov_mfma<NT>), dim3(chunks, (nt_all + 7) / 8, Z), dim3(256), 0, ctx->stream, \
                       d_y, d_x, n, dim, B0, rows_per_chunk, part)
        if (full) CROSSCOV(8, 0, full);
        switch (rest) {
        case 1: CROSSCOV(1, 128 * full, 1); break;
        case 2: CROSSCOV(2, 128 * full, 1); break;
        case 3: CROSSCOV(3, 128 * full, 1); break;
        case 4: CROSSCOV(4, 128 * full, 1); break;
        case 5: CROSSCOV(5, 128 * full, 1); break;
        case 6: CROSSCOV(6, 128 * full, 1); break;
        case 7: CROSSCOV(7, 128 * full, 1); break;
        default: break;
        }
#undef CROSSCOV
    } else {
        hipLaunchKernelGGL(vq::k_crosscov_partial, dim3(chunks), dim3(256), 0, ctx->stream, d_y, d_x,
                           n, dim, rows_per_chunk, (double *)ctx->tmp_a.p);
    }
    // chunk sums in groups of 32 chunks, then the groups
    const int per_group = 32, groups = (chunks + per_group - 1) / per_group;
    hipLaunchKernelGGL(vq::k_crosscov_reduce, dim3(cdiv(total, 256), groups), dim3(256), 0, ctx->stream,
                       (const double *)ctx->tmp_a.p, chunks, per_group, total, (double *)ctx->tmp_c.p);
    hipLaunchKernelGGL(vq::k_crosscov_reduce, dim3(cdiv(total, 256), 1), dim3(256), 0, ctx->stream,
                       (const double *)ctx->tmp_c.p, groups, groups, total, (double *)ctx->tmp_b.p);
    VQ_HIP(ctx, hipGetLastError());
    return VQ_OK;
}

}  // namespace

extern "C" {

int32_t vq_residual_sub(vq_ctx *ctx, float *d_res, int64_t n, int64_t ld, int32_t dim, int32_t k,
                        const float *d_codebook, const uint8_t *d_codes) {
    return residual_sub<uint8_t>(ctx, d_res, n, ld, dim, k, 256, d_codebook, d_codes);
}

int32_t vq_residual_sub_u16(vq_ctx *ctx, float *d_res, int64_t n, int64_t ld, int32_t dim, int32_t k,
                            const float *d_codebook, const uint16_t *d_codes) {
    return residual_sub<uint16_t>(ctx, d_res, n, ld, dim, k, 65536, d_codebook, d_codes);
}

int32_t vq_rvq_encode(vq_ctx *ctx, int32_t metric, const float *d_x, int64_t n, int64_t ld, int32_t dim,
                      int32_t stages, int32_t k, const float *d_codebooks, float epsilon, uint8_t *d_codes,
                      uint8_t *d_stages_used, uint16_t *d_recon_f16) {
    return rvq_encode<uint8_t>(ctx, metric, d_x, n, ld, dim, stages, k, 256, d_codebooks, epsilon, d_codes,
                               d_stages_used, d_recon_f16);
}

int32_t vq_rvq_encode_u16(vq_ctx *ctx, int32_t metric, const float *d_x, int64_t n, int64_t ld, int32_t dim,
                          int32_t stages, int32_t k, const float *d_codebooks, float epsilon, uint16_t *d_codes,
                          uint8_t *d_stages_used, uint16_t *d_recon_f16) {
    return rvq_encode<uint16_t>(ctx, metric, d_x, n, ld, dim, stages, k, 65536, d_codebooks, epsilon, d_codes,
                                d_stages_used, d_recon_f16);
}

int32_t vq_mean_l2norm(vq_ctx *ctx, const float *d_x, int64_t n, int64_t ld, int32_t dim, float *h_out) {
    if (!ctx) return VQ_ERR_INVALID_ARG;
    if (n == 0) return fail(ctx, VQ_ERR_EMPTY_INPUT, "Empty input: at least one vector is required.");
    if (!d_x || !h_out || n < 0 || dim <= 0 || ld < dim) return fail(ctx, VQ_ERR_INVALID_ARG, "Invalid parameter");
    VQ_HIP(ctx, hipSetDevice(ctx->device));
    const int64_t per_block = 4096;
    const int blocks = (int)cdiv(n, per_block);
    VQ_TRY(ensure(ctx, ctx->tmp_a, sizeof(float) * (size_t)n));
    VQ_TRY(ensure(ctx, ctx->tmp_b, sizeof(double) * ((size_t)blocks + 1)));
    float *norms = (float *)ctx->tmp_a.p;
    double *part = (double *)ctx->tmp_b.p;
    hipLaunchKernelGGL(vq::k_row_norms, dim3(cdiv(n, 64)), dim3(64), 0, ctx->stream, d_x, n, ld, dim, norms);
    hipLaunchKernelGGL(vq::k_sum_f64, dim3(blocks), dim3(256), 0, ctx->stream, norms,
                       (const double *)nullptr, n, per_block, part);
    hipLaunchKernelGGL(vq::k_sum_f64, dim3(1), dim3(256), 0, ctx->stream, (const float *)nullptr, part,
                       (int64_t)blocks, (int64_t)blocks, part + blocks);
    VQ_HIP(ctx, hipGetLastError());
    double total = 0.0;
    VQ_HIP(ctx, hipMemcpyAsync(&total, part + blocks, sizeof(double), hipMemcpyDeviceToHost, ctx->stream));
    VQ_HIP(ctx, hipStreamSynchronize(ctx->stream));
    *h_out = (float)total / (float)n;  // src/rvq.rs:137-138
    return VQ_OK;
}

// Up to four blocks of 32 outputs per wave of k_rotate_mfma_f32, the same number in every wave (the last ones overlap), fewer
// where that leaves compute units without rows.
static int rotate_blocks_per_wave(int64_t n, int32_t dim) {
    const int blocks = (int)cdiv(dim, 32);
    int per = 4;
    while (per > 1 && (int64_t)cdiv(n, 128) * cdiv(blocks, per) < 256) per /= 2;
    return (int)cdiv(blocks, cdiv(blocks, per));
}

// The rotation by the kernels that bf16 and the dimension ask for.
static int32_t rotate_rows(vq_ctx *ctx, const float *d_x, int64_t n, int64_t ld, int32_t dim, const float *d_R, float *d_y, bool bf16) {
    if (bf16) {
        // operand table: 32 bytes per (output dimension, 4 input dimensions)
        VQ_TRY(ensure(ctx, ctx->tmp_f, 8 * (size_t)dim * dim));
        vq::rot_u32x4 *rtab = (vq::rot_u32x4 *)ctx->tmp_f.p;
        hipLaunchKernelGGL(vq::k_rotate_prep, dim3(cdiv((int64_t)dim * dim / 4, 256)), dim3(256), 0, ctx->stream,
                           d_R, dim, rtab);
        // dim <= 128: the table (dim / 32 x 32 KB) stays in LDS, one workgroup per compute unit
#define ROTATE_RESIDENT(NB, TILES)                                                                              \
    do {                                                                                                        \
        const size_t lds = (size_t)NB * 32 * 1024;                                                              \
        auto kern = vq::k_rotate_mfma_resident<NB, TILES>;                                                      \
        VQ_HIP(ctx, hipFuncSetAttribute(reinterpret_cast<const void *>(kern),                                   \
                                        hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));                 \
        hipDeviceProp_t prop;                                                                                   \
        VQ_HIP(ctx, hipGetDeviceProperties(&prop, ctx->device));                                                \
        const int64_t groups = cdiv(n, 32 * TILES);                                                             \
        const unsigned wgs = (unsigned)std::min<int64_t>(prop.multiProcessorCount, cdiv(groups, 8));            \
        hipLaunchKernelGGL(kern, dim3(wgs), dim3(512), lds, ctx->stream, d_x, n, ld,                            \
                           (const vq::rot_u32x4 *)rtab, d_y);                                                   \
    } while (0)
#define ROTATE(NB, TILES)                                                                                    \
    hipLaunchKernelGGL((vq::k_rotate_mfma<NB, TILES>), dim3(cdiv(n, 128 * TILES)), dim3(256), 0, ctx->stream, \
                       d_x, n, ld, (const vq::rot_u32x4 *)rtab, d_y)
        switch (dim / 32) {
        case 1: ROTATE_RESIDENT(1, 2); break;
        case 2: ROTATE_RESIDENT(2, 2); break;
        case 3: ROTATE_RESIDENT(3, 2); break;
        case 4: ROTATE_RESIDENT(4, 2); break;
        case 5: ROTATE(5, 1); break;
        case 6: ROTATE(6, 1); break;
        case 7: ROTATE(7, 1); break;
        default: ROTATE(8, 1); break;
        }
#undef ROTATE
#undef ROTATE_RESIDENT
        VQ_HIP(ctx, hipGetLastError());
        return VQ_OK;
    }
    if (dim <= 3) {
        auto *kern = dim == 1 ? vq::k_rotate_narrow<1> : dim == 2 ? vq::k_rotate_narrow<2> : vq::k_rotate_narrow<3>;
        hipLaunchKernelGGL(kern, dim3(cdiv(n, 256)), dim3(256), 0, ctx->stream, d_x, n, ld, d_R, d_y);
        VQ_HIP(ctx, hipGetLastError());
        return VQ_OK;
    }
    if (dim <= 32) {
        const int nk = (int)cdiv(dim, 8);
        auto *kern = nk == 1 ? vq::k_rotate_mfma_small<1> : nk == 2 ? vq::k_rotate_mfma_small<2> : nk == 3 ? vq::k_rotate_mfma_small<3> : vq::k_rotate_mfma_small<4>;
        hipLaunchKernelGGL(kern, dim3(cdiv(n, 128)), dim3(256), 0, ctx->stream, d_x, n, ld, dim, d_R, d_y);
        VQ_HIP(ctx, hipGetLastError());
        return VQ_OK;
    }
    const int blocks = (int)cdiv(dim, 32), per = rotate_blocks_per_wave(n, dim);
    const unsigned groups = cdiv(blocks, per);
    const int entries = (int)cdiv(dim, 8) * blocks * 64;
    VQ_TRY(ensure(ctx, ctx->tmp_f, sizeof(float4) * (size_t)entries));
    float4 *rtab = (float4 *)ctx->tmp_f.p;
    hipLaunchKernelGGL(vq::k_rotate_prep_f32, dim3(cdiv(entries, 256)), dim3(256), 0, ctx->stream, d_R, dim, blocks, entries, rtab);
    auto *kern = per == 1 ? vq::k_rotate_mfma_f32<1> : per == 2 ? vq::k_rotate_mfma_f32<2> : per == 3 ? vq::k_rotate_mfma_f32<3> : vq::k_rotate_mfma_f32<4>;
    hipLaunchKernelGGL(kern, dim3(cdiv(n, 128), groups), dim3(256), 0, ctx->stream, d_x, n, ld, dim, blocks, (const float4 *)rtab, d_y);
    VQ_HIP(ctx, hipGetLastError());
    return VQ_OK;
}

int32_t vq_rotate(vq_ctx *ctx, const float *d_x, int64_t n, int64_t ld, int32_t dim, const float *d_R,
                  float *d_y) {
    if (!ctx) return VQ_ERR_INVALID_ARG;
    if (n == 0) return VQ_OK;
    if (!d_x || !d_R || !d_y || n < 0 || dim <= 0 || ld < dim) return fail(ctx, VQ_ERR_INVALID_ARG, "Invalid parameter");
    VQ_HIP(ctx, hipSetDevice(ctx->device));
    // bf16 matrix cores: dim a multiple of 32 up to 256, rows and output 16-byte aligned
    const bool bf16 = dim % 32 == 0 && dim <= 256 && ld % 4 == 0 &&
                      ((reinterpret_cast<uintptr_t>(d_x) | reinterpret_cast<uintptr_t>(d_y)) & 15) == 0;
    if (!bf16 && dim > 639) return fail(ctx, VQ_ERR_UNSUPPORTED, "rotation: dim %d too large", dim);
    // An output over the rows: a wave reads all of its rows before it writes, so compact rows may be replaced by their own
    // results where one wave makes all outputs of a row; else an output lies over rows that other waves still read.
    const bool overlap = d_y < d_x + (n - 1) * ld + dim && d_x < d_y + n * (int64_t)dim;
    const bool own = d_x == d_y && ld == dim && (bf16 || rotate_blocks_per_wave(n, dim) * 32 >= dim);
    if (!overlap || own) return rotate_rows(ctx, d_x, n, ld, dim, d_R, d_y, bf16);
    // An output that begins no later than the rows reaches none behind the ones it is made of: a slice is copied at a time
    // (64 MB).  Else all rows are, and a large copy is given back.
    const int64_t slice = d_y <= d_x ? std::min<int64_t>(n, (64 << 20) / (int64_t)sizeof(float) / dim) : n;
    VQ_TRY(ensure(ctx, ctx->tmp_e, sizeof(float) * (size_t)slice * dim));
    int32_t rc = VQ_OK;
    for (int64_t r0 = 0; r0 < n && rc == VQ_OK; r0 += slice) {
        const int64_t rows = std::min(slice, n - r0);
        VQ_HIP(ctx, hipMemcpy2DAsync(ctx->tmp_e.p, sizeof(float) * dim, d_x + r0 * ld, sizeof(float) * ld, sizeof(float) * dim,
                                     (size_t)rows, hipMemcpyDeviceToDevice, ctx->stream));
        rc = rotate_rows(ctx, (const float *)ctx->tmp_e.p, rows, dim, dim, d_R, d_y + r0 * dim, bf16);
    }
    if (ctx->tmp_e.cap > kPadKeep) {
        const int32_t gone = release(ctx, ctx->tmp_e);
        if (rc == VQ_OK) rc = gone;
    }
    return rc;
}

int32_t vq_cross_cov(vq_ctx *ctx, const float *d_y, const float *d_x, int64_t n, int32_t dim, double *h_A) {
    if (!ctx) return VQ_ERR_INVALID_ARG;
    if (n == 0) return fail(ctx, VQ_ERR_EMPTY_INPUT, "Empty input: at least one vector is required.");
    if (!d_y || !d_x || !h_A || n < 0 || dim <= 0) return fail(ctx, VQ_ERR_INVALID_ARG, "Invalid parameter");
    if (dim > 4096) return fail(ctx, VQ_ERR_UNSUPPORTED, "cross-covariance: dim %d > 4096", dim);
    VQ_HIP(ctx, hipSetDevice(ctx->device));
    VQ_TRY(cross_cov_device(ctx, d_y, d_x, n, dim));
    const size_t total = (size_t)dim * dim;
    VQ_HIP(ctx, hipMemcpyAsync(h_A, ctx->tmp_b.p, sizeof(double) * total, hipMemcpyDeviceToHost, ctx->stream));
    VQ_HIP(ctx, hipStreamSynchronize(ctx->stream));
    return VQ_OK;
}

int32_t vq_opq_rotation(vq_ctx *ctx, const float *d_y, const float *d_x, int64_t n, int32_t dim, float *d_R) {
    if (!ctx) return VQ_ERR_INVALID_ARG;
    if (n == 0) return fail(ctx, VQ_ERR_EMPTY_INPUT, "Empty input: at least one vector is required.");
    if (!d_y || !d_x || !d_R || n < 0 || dim <= 0) return fail(ctx, VQ_ERR_INVALID_ARG, "Invalid parameter");
    if (dim > 4096) return fail(ctx, VQ_ERR_UNSUPPORTED, "cross-covariance: dim %d > 4096", dim);
    VQ_HIP(ctx, hipSetDevice(ctx->device));
    hipStream_t st = ctx->stream;
    VQ_TRY(cross_cov_device(ctx, d_y, d_x, n, dim));
    const size_t total = (size_t)dim * dim;
    if (dim <= vq::kPolarMaxDim && ctx->procrustes_path == 0) {
        const int P = (dim + 15) / 16 * 16, strips = P / 16;
        const double *A = (const double *)ctx->tmp_b.p;
        VQ_TRY(ensure(ctx, ctx->tmp_a, sizeof(double) * (size_t)P * P));
        VQ_TRY(ensure(ctx, ctx->tmp_d, sizeof(double) * (size_t)P * P));
        VQ_TRY(ensure(ctx, ctx->tmp_c, sizeof(double) * (size_t)(strips + 2) * dim));
        VQ_TRY(ensure(ctx, ctx->tmp_f, 1024));
        VQ_TRY(ensure_pinned(ctx, ctx->lbg_pin, ctx->lbg_pin_cap, sizeof(int)));
        double *X[2] = {(double *)ctx->tmp_a.p, (double *)ctx->tmp_d.p};
        double *col_part = (double *)ctx->tmp_c.p, *row_sum = col_part + (size_t)strips * dim, *row_sq = row_sum + dim;
        vq::PolarTables tb;
        tb.errs = (unsigned long long *)ctx->tmp_f.p;
        tb.fin = (int *)(tb.errs + vq::kPolarMaxSteps);
        tb.bad = tb.fin + vq::kPolarMaxSteps + 2;
        static_assert(sizeof(unsigned long long) * vq::kPolarMaxSteps + sizeof(int) * (vq::kPolarMaxSteps + 3) <= 1024,
                      "step tables");
        volatile int *status = (volatile int *)ctx->lbg_pin;
        hipLaunchKernelGGL(vq::k_polar_norms, dim3(strips), dim3(256), 0, st, A, dim, col_part, row_sum, row_sq);
        hipLaunchKernelGGL(vq::k_polar_start, dim3(strips), dim3(256), 0, st, A, dim, P, (const double *)col_part,
                           (const double *)row_sum, (const double *)row_sq, tb, X[0]);
        double low = 1e-3;
        for (int s = 0; s < vq::kPolarMaxSteps;) {
            const int upto = std::min(vq::kPolarMaxSteps, s == 0 ? 16 : s + 6);
            VQ_TRY(polar_steps(ctx, X, dim, s, upto, low, tb.errs, tb.fin));
            s = upto;
            hipLaunchKernelGGL(vq::k_polar_finish, dim3(cdiv((int64_t)total, 1024)), dim3(256), 0, st,
                               (const double *)X[0], (const double *)X[1], P, dim, tb, s, d_R, (int *)ctx->lbg_pin);
            VQ_HIP(ctx, hipGetLastError());
            VQ_HIP(ctx, hipStreamSynchronize(st));
            if (*status > 0) return VQ_OK;
            if (*status < 0) break;
        }
    }
    // the SVD, from host memory
    std::vector<double> A(total), R(total);
    VQ_HIP(ctx, hipMemcpyAsync(A.data(), ctx->tmp_b.p, sizeof(double) * total, hipMemcpyDeviceToHost, st));
    VQ_HIP(ctx, hipStreamSynchronize(st));
    for (double &v : A) v = (double)(float)v;
    VQ_TRY(procrustes_svd(ctx, A.data(), dim, R.data()));
    std::vector<float> r(R.begin(), R.end());
    VQ_HIP(ctx, hipMemcpyAsync(d_R, r.data(), sizeof(float) * total, hipMemcpyHostToDevice, st));
    VQ_HIP(ctx, hipStreamSynchronize(st));
    return VQ_OK;
}

int32_t vq_ctx_set_procrustes_path(vq_ctx *ctx, int32_t path) {
    if (!ctx || (path != 0 && path != 1)) return VQ_ERR_INVALID_ARG;
    ctx->procrustes_path = path;
    return VQ_OK;
}

int32_t vq_procrustes_rotation(vq_ctx *ctx, const double *h_A, int32_t dim, double *h_R) {
    if (!ctx) return VQ_ERR_INVALID_ARG;
    if (!h_A || !h_R || dim < 1) return fail(ctx, VQ_ERR_INVALID_ARG, "Invalid parameter");
    if (dim > 4096) return fail(ctx, VQ_ERR_UNSUPPORTED, "rotation update: dim %d above 4096", dim);
    // First the polar factor by Newton-Schulz steps on the f64 matrix cores (any dim up to 512); a
    // matrix that does not converge there — singular, badly conditioned, non-finite — takes the
    // one-sided Jacobi SVD: on the device for even dim up to 128, else the same routine on the host
    // (the reference runs its SVD on the host as well, src/opq.rs:180).
    if (dim > vq::kPolarMaxDim && (dim > vq::kJacobiMax || dim % 2 != 0)) {
        vqh::procrustes_host(h_A, (size_t)dim, h_R);
        return VQ_OK;
    }
    VQ_HIP(ctx, hipSetDevice(ctx->device));
    if (ctx->procrustes_path == 0) {
        bool done = false;
        VQ_TRY(polar_newton_schulz(ctx, h_A, dim, h_R, &done));
        if (done) return VQ_OK;
    }
    return procrustes_svd(ctx, h_A, dim, h_R);
}

}  // extern "C"

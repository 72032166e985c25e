// libvqhip — codebooks of more than 256 centroids: 16-bit codes (declared in include/vq_hip.h).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstring>
#include <vector>

#include <rocprim/device/device_radix_sort.hpp>

#include "ctx.hpp"
#include "lbg_update.hpp"
#include "bigk.hpp"
#include "assign_mfma_lds.hpp"

using namespace vqh;

namespace {

constexpr int64_t kSlicePairs = 16 << 20;  // pairs assigned chunk by chunk at a time

template <int METRIC>
void launch_merge(vq_ctx *ctx, const float *d_x, int64_t n, int64_t ld, int m, int sd, int k, const float *chunks,
                  int base, int count, const uint8_t *win, const float *win_d, int64_t stride, unsigned have_d,
                  float *best, uint16_t *out) {
    hipLaunchKernelGGL(vq::k_chunk_merge<METRIC>, dim3(cdiv(n * m, 256)), dim3(256), 0, ctx->stream, d_x, n, ld, m, sd,
                       k, chunks, base, count, win, win_d, stride, have_d, best, out);
}

// Column blocks of 8 or 16 floats: the whole codebook in one pass over the rows.
int32_t launch_big(vq_ctx *ctx, int metric, const float *d_x, int64_t n, int64_t ld, int m, int sd, int k, const float *d_codebooks,
                   uint16_t *d_codes) {
    vq::LdsArgs args{};
    args.a.x = d_x;
    args.a.n = n;
    args.a.ld = ld;
    args.a.m = m;
    args.a.k = k;
    args.a.cb = d_codebooks;
    args.codes16 = d_codes;
    VQ_TRY(next_counters(ctx, &args.stat, &args.stat_next));
#define BIG(M) \
    VQ_HIP(ctx, sd == 8 ? (vq::launch_mfma_lds<M, 8, vq::CODES_U16>(ctx->stream, args)) : (vq::launch_mfma_lds<M, 16, vq::CODES_U16>(ctx->stream, args)))
    switch (metric) {
    case VQ_SQEUCLIDEAN: BIG(vq::M_SQ); break;
    case VQ_EUCLIDEAN: BIG(vq::M_EUCLID); break;
    default: BIG(vq::M_COS); break;
    }
#undef BIG
    return VQ_OK;
}

// Blocks of 8 or 16 floats in one pass, blocks of a width that an encode pads padded first (a slice of rows at a time).
// *done: it ran.
int32_t assign_big(vq_ctx *ctx, int metric, const float *d_x, int64_t n, int64_t ld, int m, int sd, int k,
                   const float *d_codebooks, uint16_t *d_codes, bool *done) {
    *done = false;
    if (ctx->assign_path == 1 || metric == VQ_MANHATTAN) return VQ_OK;
    auto fits = [&](int w) { return w == 8 ? k <= vq::kBig8Max : w == 16 && k <= vq::kLds16Max; };
    // float4 centroid loads; 32 rows within 32-bit byte offsets
    if (fits(sd) && (reinterpret_cast<uintptr_t>(d_codebooks) & 15) == 0 && ld <= (1 << 20)) {
        *done = true;
        return launch_big(ctx, metric, d_x, n, ld, m, sd, k, d_codebooks, d_codes);
    }
    const int sdp = encode_pad_width(ctx, metric, d_x, n, ld, m, sd, vq::kChunk, d_codebooks);
    if (!sdp) return VQ_OK;
    *done = true;
    const int64_t row_bytes = (int64_t)sizeof(float) * m * sdp;
    const int64_t slice = std::min<int64_t>(n, std::max<int64_t>(4096, kPadSlice / row_bytes / 4096 * 4096));
    VQ_TRY(ensure(ctx, ctx->pad_x, (size_t)(slice * row_bytes)));
    VQ_TRY(ensure(ctx, ctx->pad_cb, sizeof(float) * (size_t)m * k * sdp));
    float *px = (float *)ctx->pad_x.p, *pcb = (float *)ctx->pad_cb.p;
    pad_blocks(ctx, d_codebooks, (int64_t)m * k, sd, 1, sd, sdp, pcb);
    struct Held {  // the chunks of a slice never pad into the buffer that they read
        bool &on;
        explicit Held(bool &b) : on(b) { on = true; }
        ~Held() { on = false; }
    } held{ctx->pad_held};
    for (int64_t r0 = 0; r0 < n; r0 += slice) {
        const int64_t rows = std::min(slice, n - r0);
        pad_blocks(ctx, d_x + r0 * ld, rows, ld, m, sd, sdp, px);
        if (fits(sdp))
            VQ_TRY(launch_big(ctx, metric, px, rows, (int64_t)m * sdp, m, sdp, k, pcb, d_codes + r0 * m));
        else  // chunk by chunk
            VQ_TRY(assign_codes_u16(ctx, metric, px, rows, (int64_t)m * sdp, m, sdp, k, pcb, d_codes + r0 * m, nullptr, nullptr));
    }
    VQ_HIP(ctx, hipGetLastError());
    return VQ_OK;
}

}  // namespace

namespace vqh {

int32_t assign_codes_u16(vq_ctx *ctx, int32_t metric, const float *d_x, int64_t n, int64_t ld, int32_t m,
                         int32_t sd, int32_t k, const float *d_codebooks, uint16_t *d_codes, uint16_t *d_out16,
                         bool *out_written) {
    if (out_written) *out_written = false;
    VQ_TRY(check_common(ctx, d_x, n, ld, m, sd, k, 65536));
    if (!d_codebooks || !d_codes) return fail(ctx, VQ_ERR_INVALID_ARG, "Invalid parameter: null pointer");
    if (reinterpret_cast<uintptr_t>(d_codes) & 1)
        return fail(ctx, VQ_ERR_INVALID_ARG, "Invalid parameter: d_codes must be 2-byte aligned");
    if (m > 65535) return fail(ctx, VQ_ERR_UNSUPPORTED, "m must be at most 65535");
    if (metric < VQ_SQEUCLIDEAN || metric > VQ_MANHATTAN)
        return fail(ctx, VQ_ERR_UNSUPPORTED, "metric %d has no kernel", metric);
    VQ_HIP(ctx, hipSetDevice(ctx->device));
    if (assign_few_applicable(ctx, n, m, sd)) {
        if (out_written) *out_written = d_out16 != nullptr;
        return assign_few<uint16_t>(ctx, metric, d_x, n, ld, m, sd, k, d_codebooks, d_codes, d_out16);
    }
    if (k <= vq::kChunk) {  // one chunk: its winner is the answer
        const size_t pairs = (size_t)n * m;
        VQ_TRY(ensure(ctx, ctx->big_win, pairs));
        uint8_t *win = (uint8_t *)ctx->big_win.p;
        VQ_TRY(assign_codes(ctx, metric, d_x, n, ld, m, sd, k, d_codebooks, win));
        hipLaunchKernelGGL(vq::k_widen_codes, dim3(cdiv((int64_t)pairs, 256)), dim3(256), 0, ctx->stream,
                           (const uint8_t *)win, (int64_t)pairs, d_codes);
        VQ_HIP(ctx, hipGetLastError());
        return VQ_OK;
    }
    bool done = false;
    VQ_TRY(assign_big(ctx, metric, d_x, n, ld, m, sd, k, d_codebooks, d_codes, &done));
    if (done) return VQ_OK;
    // The rows in slices of up to kSlicePairs (row, block) pairs: the chunks that one launch merges have their
    // winners and distances side by side, 24 bytes per pair for four and the running minimum, and the
    // workspace stays at 400 MB whatever n is (slices of half the size: 1,000,000 x 16 pairs, k = 1024 1.68 ->
    // 1.71 ms, k = 2048 3.28 -> 3.34; 1,000,000 x 32 blocks of 2, k = 600: 4.22 -> 3.96).
    const int chunks = (int)cdiv(k, vq::kChunk), together = std::min(chunks, vq::kMergeChunks);
    const int64_t slice = std::min<int64_t>(n, std::max<int64_t>(1, kSlicePairs / m));
    const size_t pairs = (size_t)slice * m, stride = (pairs + 255) & ~(size_t)255;
    VQ_TRY(ensure(ctx, ctx->big_chunk, sizeof(float) * (size_t)m * k * sd));
    VQ_TRY(ensure(ctx, ctx->big_win, stride * together));
    if (chunks > together) VQ_TRY(ensure(ctx, ctx->big_best, sizeof(float) * pairs));
    VQ_TRY(ensure(ctx, ctx->big_wind, sizeof(float) * stride * together));
    uint8_t *win = (uint8_t *)ctx->big_win.p;
    float *tables = (float *)ctx->big_chunk.p;
    float *best = (float *)ctx->big_best.p;
    float *wind = (float *)ctx->big_wind.p;
    hipLaunchKernelGGL(vq::k_chunk_tables, dim3(cdiv((int64_t)m * k * sd, 256)), dim3(256), 0, ctx->stream, d_codebooks,
                       m, k, sd, tables);
    VQ_HIP(ctx, hipGetLastError());
    for (int64_t r0 = 0; r0 < n; r0 += slice) {
        const int64_t rows = std::min(slice, n - r0);
        const float *x = d_x + r0 * ld;
        uint16_t *codes = d_codes + r0 * m;
        for (int c0 = 0; c0 < chunks; c0 += together) {
            const int count = std::min(together, chunks - c0), base = c0 * vq::kChunk;
            unsigned have = 0;
            for (int c = 0; c < count; ++c) {
                const int b0 = base + c * vq::kChunk, kc = std::min(vq::kChunk, k - b0);
                // the winners' distances come with the codes where the assignment kernel computes them anyway
                bool have_d = false;
                VQ_TRY(assign_codes(ctx, metric, x, rows, ld, m, sd, kc, tables + (size_t)b0 * m * sd, win + c * stride,
                                    wind + c * stride, &have_d));
                if (have_d) have |= 1u << c;
            }
#define MERGE(M) \
    launch_merge<M>(ctx, x, rows, ld, m, sd, k, tables, base, count, win, wind, (int64_t)stride, have, best, codes)
            switch (metric) {
            case VQ_SQEUCLIDEAN: MERGE(vq::M_SQ); break;
            case VQ_EUCLIDEAN: MERGE(vq::M_EUCLID); break;
            case VQ_COSINE: MERGE(vq::M_COS); break;
            default: MERGE(vq::M_L1); break;
            }
#undef MERGE
            VQ_HIP(ctx, hipGetLastError());
        }
    }
    return VQ_OK;
}

int32_t lbg_fit_big(vq_ctx *ctx, const float *d_x, int64_t n, int64_t ld, int32_t m, int32_t sd, int32_t k,
                    int32_t max_iters, const uint32_t *h_init_idx, const uint32_t *h_reseed_stream,
                    int32_t n_reseed, float *d_codebooks, int32_t *h_iters_run, int32_t *h_reseeds_used,
                    const std::function<void()> &last) {
    hipStream_t st = ctx->stream;
    const size_t pairs = (size_t)n * m;
    if (pairs >= (1ULL << 32)) return fail(ctx, VQ_ERR_UNSUPPORTED, "n * m must be below 2^32 when k is above 256");
    const int big_cap = (int)std::min<int64_t>(k, n / (vq::kBigSeqMax + 1) + 1);
    const size_t mk = (size_t)m * k;
    VQ_TRY(ensure(ctx, ctx->big_flags, sizeof(int) * (6 * (size_t)m + 1)));
    VQ_TRY(ensure(ctx, ctx->big_tables, sizeof(uint32_t) * (3 * mk + (size_t)m * big_cap)));
    VQ_TRY(ensure(ctx, ctx->big_codes, sizeof(uint16_t) * pairs));
    VQ_TRY(ensure(ctx, ctx->big_fresh, sizeof(uint16_t) * pairs));
    VQ_TRY(ensure(ctx, ctx->big_keys, sizeof(uint64_t) * pairs));
    VQ_TRY(ensure(ctx, ctx->big_sorted, sizeof(uint64_t) * pairs));
    VQ_TRY(ensure(ctx, ctx->idx, sizeof(uint32_t) * mk));
    VQ_TRY(ensure(ctx, ctx->reseed, sizeof(uint32_t) * ((size_t)m * n_reseed + 1)));
    // keys: row in bits 0-31, code in the next code_bits, column block above; they are written block by
    // block in row order, so the sort covers the bits from 32 up only (a radix sort is stable)
    int code_bits = 1;
    while ((1 << code_bits) < k) ++code_bits;
    unsigned end_bit = 32u + (unsigned)code_bits;
    while (end_bit < 64 && ((uint64_t)(m - 1) >> (end_bit - 32u - (unsigned)code_bits)) != 0) ++end_bit;
    uint64_t *keys = (uint64_t *)ctx->big_keys.p, *sorted = (uint64_t *)ctx->big_sorted.p;
    size_t sort_bytes = 0;
    VQ_HIP(ctx, rocprim::radix_sort_keys(nullptr, sort_bytes, keys, sorted, pairs, 32u, end_bit, st));
    VQ_TRY(ensure(ctx, ctx->big_sort_tmp, sort_bytes));

    vq::BigLbg S;
    int *f = (int *)ctx->big_flags.p;
    S.changed = f;
    S.done = f + m;
    S.iters = f + 2 * m;
    S.used = f + 3 * m;
    S.ubase = f + 4 * m;
    S.nbig = f + 5 * m;
    S.err = f + 6 * m;
    uint32_t *tb = (uint32_t *)ctx->big_tables.p;
    S.count = tb;
    S.start = tb + mk;
    S.empty_rank = tb + 2 * mk;
    S.big_list = tb + 3 * mk;
    S.big_cap = big_cap;
    S.codes = (uint16_t *)ctx->big_codes.p;
    uint16_t *fresh = (uint16_t *)ctx->big_fresh.p;

    VQ_HIP(ctx, hipMemcpyAsync(ctx->idx.p, h_init_idx, sizeof(uint32_t) * mk, hipMemcpyHostToDevice, st));
    if (n_reseed)
        VQ_HIP(ctx, hipMemcpyAsync(ctx->reseed.p, h_reseed_stream, sizeof(uint32_t) * (size_t)m * n_reseed,
                                   hipMemcpyHostToDevice, st));
    VQ_HIP(ctx, hipMemsetAsync(S.codes, 0, sizeof(uint16_t) * pairs, st));  // assignments = vec![0; n], utils.rs:55
    hipLaunchKernelGGL(vq::k_big_init, dim3(cdiv(m, 64)), dim3(64), 0, st, S, m);
    hipLaunchKernelGGL(vq::k_gather_rows, dim3(cdiv((int64_t)mk * sd, 256)), dim3(256), 0, st, d_x, ld, m, k, sd,
                       (const uint32_t *)ctx->idx.p, d_codebooks);
    VQ_HIP(ctx, hipGetLastError());

    std::vector<int> host(6 * (size_t)m + 1);
    for (int it = 0; it < max_iters; ++it) {
        {
            ProfSpan sp(ctx, VQ_PROF_LBG_ASSIGN);
            VQ_TRY(assign_codes_u16(ctx, VQ_SQEUCLIDEAN, d_x, n, ld, m, sd, k, d_codebooks, fresh));
        }
        ProfSpan sp(ctx, VQ_PROF_LBG_UPDATE);
        hipLaunchKernelGGL(vq::k_big_commit, dim3(cdiv(n, 256), cdiv(m, vq::kCommitBlocks)), dim3(256), 0, st, S, (const uint16_t *)fresh, n, m,
                           code_bits, keys);
        VQ_HIP(ctx, hipGetLastError());
        VQ_HIP(ctx, rocprim::radix_sort_keys(ctx->big_sort_tmp.p, sort_bytes, keys, sorted, pairs, 32u, end_bit, st));
        VQ_HIP(ctx, hipMemsetAsync(S.count, 0, sizeof(uint32_t) * mk, st));
        hipLaunchKernelGGL(vq::k_big_bounds, dim3(cdiv((int64_t)pairs, 256)), dim3(256), 0, st, S,
                           (const uint64_t *)sorted, n, m, k, code_bits);
        hipLaunchKernelGGL(vq::k_big_plan, dim3(m), dim3(256), 0, st, S, k);
        if (n >= 32 * (int64_t)k) {  // two waves per cluster and 32 components
            const int tiles = (int)cdiv(sd, 32), width = tiles == 1 ? sd : (int)cdiv(cdiv(sd, tiles), 4) * 4;
            const int vec = sd >= 4 ? 4 : 1, pieces = (int)cdiv(width, vec);
            const size_t lds = sizeof(float) * (size_t)width * (8 * (128 / pieces) + 4);
            hipLaunchKernelGGL(vec == 4 ? vq::k_big_means_tile<4> : vq::k_big_means_tile<1>, dim3(k, m, cdiv(sd, width)), dim3(128), lds, st, S,
                               (const uint64_t *)sorted, d_x, n, ld, k, sd, width, pieces, (const uint32_t *)ctx->reseed.p,
                               n_reseed, d_codebooks);
        } else {
            hipLaunchKernelGGL(vq::k_big_small_means, dim3(cdiv((int64_t)k * sd, 256), m), dim3(256), 0, st, S,
                               (const uint64_t *)sorted, d_x, n, ld, k, sd, (const uint32_t *)ctx->reseed.p, n_reseed,
                               d_codebooks);
        }
        hipLaunchKernelGGL(vq::k_big_large_means, dim3(big_cap, m), dim3(256), 0, st, S, (const uint64_t *)sorted, d_x,
                           n, ld, k, sd, d_codebooks);
        hipLaunchKernelGGL(vq::k_big_advance, dim3(cdiv(m, 64)), dim3(64), 0, st, S, m);
        if (last && it == max_iters - 1) last();
        VQ_HIP(ctx, hipGetLastError());
        // every column block converged (src/utils.rs:104-106): the remaining passes would change nothing
        VQ_HIP(ctx, hipMemcpyAsync(host.data(), f, sizeof(int) * host.size(), hipMemcpyDeviceToHost, st));
        VQ_HIP(ctx, hipStreamSynchronize(st));
        bool all_done = true;
        for (int s = 0; s < m; ++s) all_done = all_done && host[(size_t)m + s] != 0;
        if (all_done || host[6 * (size_t)m]) {
            if (last && it < max_iters - 1) {
                last();
                VQ_HIP(ctx, hipGetLastError());
                VQ_HIP(ctx, hipStreamSynchronize(st));
            }
            break;
        }
    }
    if (max_iters == 0) {
        VQ_HIP(ctx, hipMemcpyAsync(host.data(), f, sizeof(int) * host.size(), hipMemcpyDeviceToHost, st));
        VQ_HIP(ctx, hipStreamSynchronize(st));
    }
    prof_collect(ctx);
    if (h_iters_run) memcpy(h_iters_run, host.data() + 2 * (size_t)m, sizeof(int) * m);
    if (h_reseeds_used) memcpy(h_reseeds_used, host.data() + 3 * (size_t)m, sizeof(int) * m);
    if (host[6 * (size_t)m])
        return fail(ctx, VQ_ERR_RESEED_EXHAUSTED, "re-seed stream exhausted: pass n_reseed = k*max_iters");
    return VQ_OK;
}

}  // namespace vqh

extern "C" {

int32_t vq_assign_u16(vq_ctx *ctx, int32_t metric, const float *d_x, int64_t n, int64_t ld, int32_t m, int32_t sd,
                      int32_t k, const float *d_codebooks, uint16_t *d_codes) {
    return vqh::assign_codes_u16(ctx, metric, d_x, n, ld, m, sd, k, d_codebooks, d_codes);
}

}  // extern "C"

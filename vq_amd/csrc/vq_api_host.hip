// libvqhip — copies between host and device memory, batches of host rows (declared in include/vq_hip.h).
#include <hip/hip_runtime.h>

#include "ctx.hpp"
#include "host_batch.hpp"

namespace {

// Page-locked memory and device memory by a kernel: for copies too short for the copy engine, whose
// start alone takes longer (16-byte aligned buffers, sizes rounded up to 16 bytes).
__global__ void __launch_bounds__(256) k_copy16(const uint4 *__restrict__ src, uint4 *__restrict__ dst, int64_t count) {
    const int64_t stride = (int64_t)gridDim.x * 256;
    for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < count; i += stride) dst[i] = src[i];
}

constexpr size_t kKernelCopy = 1u << 20;    // copies up to here go by kernel, batches up to here as one chunk
constexpr size_t kDirectRows = 4u << 10;    // rows up to here are read in place
constexpr size_t kPiece = 256u << 10;       // of a chunk, per claim of a copying thread

size_t up16(size_t b) { return (b + 15) & ~(size_t)15; }
size_t up256(size_t b) { return (b + 255) & ~(size_t)255; }

int32_t move(vq_ctx *ctx, void *dst, const void *src, size_t bytes, hipMemcpyKind kind, hipStream_t st) {
    if (bytes <= kKernelCopy) {
        const int64_t count = (int64_t)(up16(bytes) / 16);
        hipLaunchKernelGGL(k_copy16, dim3(std::min<unsigned>(vqh::cdiv(count, 256), 256u)), dim3(256), 0, st,
                           (const uint4 *)src, (uint4 *)dst, count);
        VQ_HIP(ctx, hipGetLastError());
    } else {
        VQ_HIP(ctx, hipMemcpyAsync(dst, src, bytes, kind, st));
    }
    return VQ_OK;
}

int32_t ensure_pipe(vq_ctx *ctx) {
    if (!ctx->up) VQ_HIP(ctx, hipStreamCreateWithFlags(&ctx->up, hipStreamNonBlocking));
    if (!ctx->down) VQ_HIP(ctx, hipStreamCreateWithFlags(&ctx->down, hipStreamNonBlocking));
    for (int i = 0; i < vq_ctx::kPipe; ++i)
        for (hipEvent_t *e : {&ctx->pipe_up[i], &ctx->pipe_run[i], &ctx->pipe_down[i]})
            if (!*e) VQ_HIP(ctx, hipEventCreateWithFlags(e, hipEventDisableTiming));
    return VQ_OK;
}

}  // namespace

namespace vqh {

CopyCrew &crew(vq_ctx *ctx) {
    if (!ctx->crew) ctx->crew = new CopyCrew;
    return *ctx->crew;
}

void drop_crew(vq_ctx *ctx) {
    delete ctx->crew;
    ctx->crew = nullptr;
}

int32_t staged_copy(vq_ctx *ctx, void *d, void *h, size_t bytes, bool upload) {
    constexpr int NB = vq_ctx::kPipe;
    // chunks short enough that the first and the last, which nothing overlaps, cost little, and long enough
    // that the gaps between the copy engine's transfers do not count (512 MB up: 11.2 ms in chunks of 4 MiB,
    // 10.2 of 8, 9.7 of 16; down 11.0, 10.1, 9.6; 128 MB up 2.9, 2.7, 2.7)
    const size_t chunk = std::min<size_t>(16u << 20, std::max<size_t>(512u << 10, up256(bytes / 8)));
    VQ_HIP(ctx, hipSetDevice(ctx->device));  // the pipeline's streams and events are made on the current device
    VQ_TRY(ensure_pipe(ctx));
    VQ_HIP(ctx, hipStreamSynchronize(ctx->stream));  // the data is there, the staging memory is idle
    VQ_TRY(ensure_pinned(ctx, ctx->pipe_pin, ctx->pipe_pin_cap, NB * chunk));
    Chunks ch(bytes, chunk, kPiece);
    char *pin = (char *)ctx->pipe_pin;
    auto slot = [&](size_t c) { return pin + (c % NB) * chunk; };
    PieceQueue q;
    q.limit.store(upload ? std::min<size_t>(NB, ch.count) * ch.per_chunk : 0);
    std::atomic<bool> quit{false};
    auto step = [&] {
        size_t p;
        if (!q.claim(p)) return false;
        ch.copy(p, (char *)h, slot, upload);
        return true;
    };
    const std::function<void()> body = [&] {
        while (!quit.load(std::memory_order_acquire))
            if (!step()) std::this_thread::yield();
    };
    CopyCrew &cr = crew(ctx);
    cr.start(crew_for(bytes), &body);
    hipError_t err = hipSuccess;
    size_t issued = 0, finished = 0;  // chunks given to the copy engine; chunks that it has moved
    while (err == hipSuccess && (upload ? finished < ch.count : finished < ch.count || !ch.complete(ch.count - 1))) {
        bool moved = false;
        const bool free_slot = issued < finished + NB;
        if (issued < ch.count && (upload ? ch.complete(issued) : free_slot && (issued < NB || ch.complete(issued - NB)))) {
            void *dp = (char *)d + issued * chunk;
            err = upload ? hipMemcpyAsync(dp, slot(issued), ch.bytes(issued), hipMemcpyHostToDevice, ctx->stream)
                         : hipMemcpyAsync(slot(issued), dp, ch.bytes(issued), hipMemcpyDeviceToHost, ctx->stream);
            if (err == hipSuccess) err = hipEventRecord(ctx->pipe_up[issued % NB], ctx->stream);
            ++issued;
            moved = true;
        }
        if (err == hipSuccess && finished < issued) {
            const hipError_t e = hipEventQuery(ctx->pipe_up[finished % NB]);
            if (e == hipSuccess) {
                ++finished;
                q.limit.store((upload ? std::min(ch.count, finished + NB) : finished) * ch.per_chunk, std::memory_order_release);
                moved = true;
            } else if (e != hipErrorNotReady) {
                err = e;
            }
        }
        if (!moved && !step()) std::this_thread::yield();
    }
    // (downloads: pieces of earlier chunks may still be under way in other threads)
    if (err == hipSuccess && !upload)
        for (size_t c = 0; c < ch.count; ++c)
            while (!ch.complete(c))
                if (!step()) std::this_thread::yield();
    quit.store(true, std::memory_order_release);
    cr.finish();
    (void)hipStreamSynchronize(ctx->stream);
    (void)hipGetLastError();
    VQ_HIP(ctx, err);
    return VQ_OK;
}

int32_t host_batch(vq_ctx *ctx, const float *h_x, int64_t n, size_t row_in, const HostOut (&outs)[2], size_t chunk_bytes,
                   bool direct, const HostRun &run) {
    constexpr int NB = vq_ctx::kPipe;
    VQ_HIP(ctx, hipSetDevice(ctx->device));
    const int64_t rows = std::min<int64_t>(n, std::max<int64_t>(1, (int64_t)(chunk_bytes / row_in)));  // per chunk
    const size_t in_b = up256(row_in * rows), o0 = up256(outs[0].row * rows), o1 = up256(outs[1].row * rows);
    const size_t slot_b = in_b + o0 + o1;
    const int slots = rows < n ? NB : 1;
    VQ_TRY(ensure_pinned(ctx, ctx->pipe_pin, ctx->pipe_pin_cap, slots * slot_b));
    char *pin = (char *)ctx->pipe_pin;
    if (direct && slots == 1 && n * row_in <= kDirectRows) {
        memcpy(pin, h_x, n * row_in);
        VQ_TRY(run((const float *)pin, n, pin + in_b, pin + in_b + o0));
        VQ_HIP(ctx, hipStreamSynchronize(ctx->stream));
        for (int o = 0; o < 2; ++o)
            if (outs[o].h) memcpy(outs[o].h, pin + in_b + (o ? o0 : 0), n * outs[o].row);
        return VQ_OK;
    }
    VQ_TRY(ensure(ctx, ctx->pipe_dev, slots * slot_b));
    char *dev = (char *)ctx->pipe_dev.p;
    if (slots == 1 && n * row_in <= kKernelCopy) {  // one chunk, the caller's thread alone, one stream
        memcpy(pin, h_x, n * row_in);
        VQ_TRY(move(ctx, dev, pin, n * row_in, hipMemcpyHostToDevice, ctx->stream));
        VQ_TRY(run((const float *)dev, n, dev + in_b, dev + in_b + o0));
        for (int o = 0; o < 2; ++o)
            if (outs[o].h) {
                const size_t at = in_b + (o ? o0 : 0);
                VQ_TRY(move(ctx, pin + at, dev + at, n * outs[o].row, hipMemcpyDeviceToHost, ctx->stream));
            }
        VQ_HIP(ctx, hipStreamSynchronize(ctx->stream));
        for (int o = 0; o < 2; ++o)
            if (outs[o].h) memcpy(outs[o].h, pin + in_b + (o ? o0 : 0), n * outs[o].row);
        return VQ_OK;
    }
    VQ_TRY(ensure_pipe(ctx));
    VQ_HIP(ctx, hipStreamSynchronize(ctx->stream));  // the slots are idle
    Chunks in(n * row_in, row_in * rows, kPiece);
    Chunks out0(n * outs[0].row, outs[0].row * rows, kPiece), out1(n * outs[1].row, outs[1].row * rows, kPiece);
    const size_t count = in.count;
    auto slot = [&](size_t c) { return pin + (c % NB) * slot_b; };
    auto slot0 = [&](size_t c) { return slot(c) + in_b; };
    auto slot1 = [&](size_t c) { return slot(c) + in_b + o0; };
    PieceQueue qi, q0, q1;
    qi.limit.store(std::min<size_t>(NB, count) * in.per_chunk);
    std::atomic<bool> quit{false};
    auto step = [&] {  // results first: they free a slot
        size_t p;
        if (q0.claim(p))
            out0.copy(p, (char *)outs[0].h, slot0, false);
        else if (q1.claim(p))
            out1.copy(p, (char *)outs[1].h, slot1, false);
        else if (qi.claim(p))
            in.copy(p, (char *)const_cast<float *>(h_x), slot, true);
        else
            return false;
        return true;
    };
    const std::function<void()> body = [&] {
        while (!quit.load(std::memory_order_acquire))
            if (!step()) std::this_thread::yield();
    };
    auto emptied = [&](size_t c) { return (!outs[0].h || out0.complete(c)) && (!outs[1].h || out1.complete(c)); };
    CopyCrew &cr = crew(ctx);
    cr.start(crew_for(n * (row_in + (outs[0].h ? outs[0].row : 0) + (outs[1].h ? outs[1].row : 0))), &body);
    // chunks whose upload and computation are enqueued; uploaded; whose download is enqueued; arrived; copied out
    size_t run_n = 0, up_n = 0, down_n = 0, here_n = 0, out_n = 0;
    int32_t rc = VQ_OK;
    auto ready = [&](hipEvent_t e) {
        const hipError_t q = hipEventQuery(e);
        if (q == hipErrorNotReady) (void)hipGetLastError();
        else if (q != hipSuccess && rc == VQ_OK) rc = fail(ctx, VQ_ERR_HIP, "host batch: %s", hipGetErrorString(q));
        return q == hipSuccess;
    };
    auto enqueue_run = [&](size_t c) -> int32_t {
        const int b = (int)(c % NB);
        char *d = dev + b * slot_b;
        if (c >= (size_t)NB) VQ_HIP(ctx, hipStreamWaitEvent(ctx->up, ctx->pipe_run[b], 0));  // the rows in this slot have been read
        VQ_TRY(move(ctx, d, slot(c), in.bytes(c), hipMemcpyHostToDevice, ctx->up));
        VQ_HIP(ctx, hipEventRecord(ctx->pipe_up[b], ctx->up));
        VQ_HIP(ctx, hipStreamWaitEvent(ctx->stream, ctx->pipe_up[b], 0));
        if (c >= (size_t)NB) VQ_HIP(ctx, hipStreamWaitEvent(ctx->stream, ctx->pipe_down[b], 0));  // its results have left
        VQ_TRY(run((const float *)d, (int64_t)(in.bytes(c) / row_in), d + in_b, d + in_b + o0));
        VQ_HIP(ctx, hipEventRecord(ctx->pipe_run[b], ctx->stream));
        return VQ_OK;
    };
    auto enqueue_down = [&](size_t c) -> int32_t {
        const int b = (int)(c % NB);
        char *d = dev + b * slot_b + in_b;
        VQ_HIP(ctx, hipStreamWaitEvent(ctx->down, ctx->pipe_run[b], 0));
        if (outs[0].h) VQ_TRY(move(ctx, slot0(c), d, out0.bytes(c), hipMemcpyDeviceToHost, ctx->down));
        if (outs[1].h) VQ_TRY(move(ctx, slot1(c), d + o0, out1.bytes(c), hipMemcpyDeviceToHost, ctx->down));
        VQ_HIP(ctx, hipEventRecord(ctx->pipe_down[b], ctx->down));
        return VQ_OK;
    };
    while (rc == VQ_OK && out_n < count) {
        bool moved = false;
        if (up_n < run_n && ready(ctx->pipe_up[up_n % NB])) {  // its staging buffer is free again
            ++up_n;
            qi.limit.store(std::min(count, up_n + NB) * in.per_chunk, std::memory_order_release);
            moved = true;
        }
        // (a slot's results are given to the copy engine before its next computation is enqueued)
        if (rc == VQ_OK && run_n < count && run_n < down_n + NB && in.complete(run_n)) {
            rc = enqueue_run(run_n++);
            moved = true;
        }
        if (rc == VQ_OK && down_n < run_n && down_n < out_n + NB) {
            rc = enqueue_down(down_n++);
            moved = true;
        }
        if (rc == VQ_OK && here_n < down_n && ready(ctx->pipe_down[here_n % NB])) {
            ++here_n;
            if (outs[0].h) q0.limit.store(here_n * out0.per_chunk, std::memory_order_release);
            if (outs[1].h) q1.limit.store(here_n * out1.per_chunk, std::memory_order_release);
            moved = true;
        }
        while (out_n < here_n && emptied(out_n)) {
            ++out_n;
            moved = true;
        }
        if (!moved && !step()) std::this_thread::yield();
    }
    quit.store(true, std::memory_order_release);
    cr.finish();
    if (rc != VQ_OK) {  // copies already enqueued read and write the slots
        (void)hipStreamSynchronize(ctx->up);
        (void)hipStreamSynchronize(ctx->down);
    }
    (void)hipStreamSynchronize(ctx->stream);
    return rc;
}

}  // namespace vqh

using namespace vqh;

// Copies of pageable memory from here on go through the staging buffers of the context, below them through
// the runtime's own path.  Up, rows that the caller has just written (an array not touched for long in
// brackets): 5 MB 0.16 ms by the runtime, 0.24 staged, 12 MB 0.34 and 0.38 (0.43 and 0.40), 20 MB 0.55 and
// 0.56 (0.75 and 0.61), 100 MB 3.5 and 2.5; down: 3 MB 0.17 and 0.18, 5 MB 0.28 and 0.25, 12 MB 0.67 and
// 0.39, 100 MB 5.9 and 2.3.
static constexpr size_t kStagedUp = 16u << 20, kStagedDown = 4u << 20;
static bool pageable(const void *h) {
    hipPointerAttribute_t attr;
    const bool locked = hipPointerGetAttributes(&attr, h) == hipSuccess && attr.type == hipMemoryTypeHost;
    (void)hipGetLastError();  // an unregistered host pointer is reported as an error: that is the pageable case
    return !locked;
}

extern "C" {

int32_t vq_h2d(vq_ctx *ctx, void *d_dst, const void *h_src, size_t bytes) {
    if (!ctx || (bytes && (!d_dst || !h_src))) return VQ_ERR_INVALID_ARG;
    if (bytes >= kStagedUp && pageable(h_src)) return staged_copy(ctx, d_dst, const_cast<void *>(h_src), bytes, true);
    VQ_HIP(ctx, hipMemcpyAsync(d_dst, h_src, bytes, hipMemcpyHostToDevice, ctx->stream));
    VQ_HIP(ctx, hipStreamSynchronize(ctx->stream));
    return VQ_OK;
}

int32_t vq_d2h(vq_ctx *ctx, void *h_dst, const void *d_src, size_t bytes) {
    if (!ctx || (bytes && (!h_dst || !d_src))) return VQ_ERR_INVALID_ARG;
    if (bytes >= kStagedDown && pageable(h_dst)) return staged_copy(ctx, const_cast<void *>(d_src), h_dst, bytes, false);
    VQ_HIP(ctx, hipMemcpyAsync(h_dst, d_src, bytes, hipMemcpyDeviceToHost, ctx->stream));
    VQ_HIP(ctx, hipStreamSynchronize(ctx->stream));
    return VQ_OK;
}

int32_t vq_pq_quantize_host(vq_ctx *ctx, int32_t metric, const float *h_x, int64_t n, int32_t m, int32_t sub_dim, int32_t k,
                            const float *d_codebooks, const float *d_rotation, void *h_codes, uint16_t *h_out) {
    if (!ctx) return VQ_ERR_INVALID_ARG;
    const int64_t dim = (int64_t)m * sub_dim;
    VQ_TRY(check_common(ctx, h_x, n, dim, m, sub_dim, k, 65536));
    if (!d_codebooks) return fail(ctx, VQ_ERR_INVALID_ARG, "Invalid parameter: null pointer");
    const bool wide = k > 256;
    const HostOut outs[2] = {{h_out, 2 * (size_t)dim}, {h_codes, (wide ? 2 : 1) * (size_t)m}};
    return host_batch(ctx, h_x, n, sizeof(float) * (size_t)dim, outs, 4u << 20, d_rotation == nullptr,
                      [&](const float *d_x, int64_t rows, void *d_out, void *d_codes) -> int32_t {
                          if (d_rotation) {
                              VQ_TRY(ensure(ctx, ctx->pipe_rot, sizeof(float) * (size_t)(rows * dim)));
                              VQ_TRY(vq_rotate(ctx, d_x, rows, dim, (int32_t)dim, d_rotation, (float *)ctx->pipe_rot.p));
                              d_x = (const float *)ctx->pipe_rot.p;
                          }
                          bool have = false;
                          if (wide)
                              VQ_TRY(assign_codes_u16(ctx, metric, d_x, rows, dim, m, sub_dim, k, d_codebooks, (uint16_t *)d_codes,
                                                      h_out ? (uint16_t *)d_out : nullptr, &have));
                          else
                              VQ_TRY(assign_codes(ctx, metric, d_x, rows, dim, m, sub_dim, k, d_codebooks, (uint8_t *)d_codes,
                                                  nullptr, nullptr, nullptr, h_out ? (uint16_t *)d_out : nullptr, &have));
                          if (!h_out || have) return VQ_OK;
                          return wide ? vq_decode_f16_u16(ctx, (const uint16_t *)d_codes, rows, m, sub_dim, k, d_codebooks, (uint16_t *)d_out)
                                      : vq_decode_f16(ctx, (const uint8_t *)d_codes, rows, m, sub_dim, k, d_codebooks, (uint16_t *)d_out);
                      });
}

int32_t vq_rvq_quantize_host(vq_ctx *ctx, int32_t metric, const float *h_x, int64_t n, int32_t dim, int32_t stages, int32_t k,
                             const float *d_codebooks, float epsilon, void *h_codes, uint16_t *h_out) {
    if (!ctx) return VQ_ERR_INVALID_ARG;
    if (n == 0) return VQ_OK;
    if (!h_x || !d_codebooks || n < 0 || dim <= 0 || stages < 0 || k <= 0)
        return fail(ctx, VQ_ERR_INVALID_ARG, "Invalid parameter");
    const bool wide = k > 256;
    const HostOut outs[2] = {{h_out, 2 * (size_t)dim}, {stages ? h_codes : nullptr, (wide ? 2 : 1) * (size_t)std::max(stages, 1)}};
    // (chunks large enough for the stages' launches)
    return host_batch(ctx, h_x, n, sizeof(float) * (size_t)dim, outs, 16u << 20, true,
                      [&](const float *d_x, int64_t rows, void *d_out, void *d_codes) -> int32_t {
                          return wide ? vq_rvq_encode_u16(ctx, metric, d_x, rows, dim, dim, stages, k, d_codebooks, epsilon,
                                                          (uint16_t *)d_codes, nullptr, h_out ? (uint16_t *)d_out : nullptr)
                                      : vq_rvq_encode(ctx, metric, d_x, rows, dim, dim, stages, k, d_codebooks, epsilon,
                                                      (uint8_t *)d_codes, nullptr, h_out ? (uint16_t *)d_out : nullptr);
                      });
}

}  // extern "C"

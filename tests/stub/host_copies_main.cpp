// The library's host-side copies and batches (vq_amd/csrc/vq_api_host.hip, host_batch.hpp: the copying
// threads, the staged copies, the pipeline of host rows) on the CPU against the stand-in runtime of
// cpu_hip/, for builds under the thread and the address sanitizers.  The computation of a batch is a
// function of the row that any order or mix-up of chunks would show.  Prints "host copies: ok" and returns 0.
#include <cstdio>
#include <vector>

#include "../../vq_amd/csrc/vq_api_host.hip"

static int failures = 0;
#define CHECK(cond)                                                         \
    do {                                                                    \
        if (!(cond)) {                                                      \
            std::fprintf(stderr, "%s:%d: %s\n", __FILE__, __LINE__, #cond); \
            ++failures;                                                     \
        }                                                                   \
    } while (0)

// ---- what the entry points call, on the context's stream ---------------------------------------
static std::atomic<int> runs{0}, fail_run_at{0};  // launches of a computation; the one that is to fail (0: none)

static uint16_t code_of(float x, int k) { return (uint16_t)((int)x % k); }
static uint16_t half_of(float x, uint16_t code) { return (uint16_t)(3 * (int)x + code); }

template <class CodeT>
static int32_t encode(vq_ctx *ctx, const float *x, int64_t n, int64_t ld, int m, int sd, int k, CodeT *codes, uint16_t *out) {
    if (++runs == fail_run_at) return fail(ctx, VQ_ERR_UNSUPPORTED, "asked to fail");
    ctx->stream->push([=] {
        for (int64_t i = 0; i < n; ++i)
            for (int s = 0; s < m; ++s) {
                const CodeT c = (CodeT)code_of(x[i * ld + s * sd], k);
                codes[i * m + s] = c;
                for (int t = 0; out && t < sd; ++t) out[(i * m + s) * sd + t] = half_of(x[i * ld + s * sd + t], c);
            }
    });
    return VQ_OK;
}
namespace vqh {
std::string &create_error() {
    static std::string e;
    return e;
}
int32_t check_common(vq_ctx *ctx, const void *x, int64_t n, int64_t, int32_t, int32_t, int32_t, int32_t) {
    return x && n > 0 ? VQ_OK : fail(ctx, VQ_ERR_INVALID_ARG, "Invalid parameter");
}
int32_t assign_codes(vq_ctx *ctx, int32_t, const float *x, int64_t n, int64_t ld, int32_t m, int32_t sd, int32_t k,
                     const float *, uint8_t *codes, float *, bool *, const PendingUpdate *, uint16_t *out, bool *written) {
    *written = out != nullptr;
    return encode(ctx, x, n, ld, m, sd, k, codes, out);
}
int32_t assign_codes_u16(vq_ctx *ctx, int32_t, const float *x, int64_t n, int64_t ld, int32_t m, int32_t sd, int32_t k,
                         const float *, uint16_t *codes, uint16_t *out, bool *written) {
    *written = out != nullptr;
    return encode(ctx, x, n, ld, m, sd, k, codes, out);
}
}  // namespace vqh
extern "C" {
int32_t vq_rotate(vq_ctx *ctx, const float *x, int64_t n, int64_t ld, int32_t dim, const float *, float *y) {
    ctx->stream->push([=] {
        for (int64_t i = 0; i < n * dim; ++i) y[i] = x[i / dim * ld + i % dim] + 1.0f;
    });
    return VQ_OK;
}
int32_t vq_decode_f16(vq_ctx *, const uint8_t *, int64_t, int32_t, int32_t, int32_t, const float *, uint16_t *) { std::abort(); }
int32_t vq_decode_f16_u16(vq_ctx *, const uint16_t *, int64_t, int32_t, int32_t, int32_t, const float *, uint16_t *) { std::abort(); }
int32_t vq_rvq_encode(vq_ctx *ctx, int32_t, const float *x, int64_t n, int64_t ld, int32_t dim, int32_t stages, int32_t k,
                      const float *, float, uint8_t *codes, uint8_t *, uint16_t *out) {
    return encode(ctx, x, n, ld, stages, dim / stages, k, codes, out);
}
int32_t vq_rvq_encode_u16(vq_ctx *ctx, int32_t, const float *x, int64_t n, int64_t ld, int32_t dim, int32_t stages, int32_t k,
                          const float *, float, uint16_t *codes, uint8_t *, uint16_t *out) {
    return encode(ctx, x, n, ld, stages, dim / stages, k, codes, out);
}
}

// ---- a context as vq_ctx_create makes it ---------------------------------------------------------
static vq_ctx *open_ctx(int device) {
    vq_ctx *ctx = new vq_ctx;
    ctx->device = device;
    (void)hipSetDevice(device);
    (void)hipStreamCreateWithFlags(&ctx->stream, 0);
    return ctx;
}
static void close_ctx(vq_ctx *ctx) {
    (void)hipStreamSynchronize(ctx->stream);
    drop_crew(ctx);
    if (ctx->pipe_pin) (void)hipHostFree(ctx->pipe_pin);
    for (DevBuf *b : {&ctx->pipe_dev, &ctx->pipe_rot})
        if (b->p) (void)hipFree(b->p);
    for (int i = 0; i < vq_ctx::kPipe; ++i)
        for (hipEvent_t e : {ctx->pipe_up[i], ctx->pipe_run[i], ctx->pipe_down[i]})
            if (e) (void)hipEventDestroy(e);
    for (hipStream_t s : {ctx->up, ctx->down, ctx->stream})
        if (s) (void)hipStreamDestroy(s);
    delete ctx;
}

static std::vector<uint8_t> pattern(size_t bytes, unsigned seed) {
    std::vector<uint8_t> v(bytes);
    uint32_t s = seed * 2654435761u + 1u;
    for (uint8_t &b : v) b = (uint8_t)((s = s * 1664525u + 1013904223u) >> 24);
    return v;
}

static void copy_there_and_back(vq_ctx *ctx, size_t bytes) {
    const std::vector<uint8_t> h = pattern(bytes, (unsigned)bytes);
    std::vector<uint8_t> back(bytes, 0xAB), dev(bytes);
    CHECK(vq_h2d(ctx, dev.data(), h.data(), bytes) == VQ_OK);
    CHECK(dev == h);
    CHECK(vq_d2h(ctx, back.data(), dev.data(), bytes) == VQ_OK);
    CHECK(back == h);
}

// n rows of m * sd floats through vq_pq_quantize_host (rotation: one is added to every component)
static void batch(vq_ctx *ctx, int64_t n, int m, int sd, int k, bool rotation, bool codes, bool out) {
    const int dim = m * sd;
    std::vector<float> x((size_t)n * dim);
    for (size_t i = 0; i < x.size(); ++i) x[i] = (float)((i * 7 + i / dim) % 1000);
    std::vector<uint8_t> c((size_t)n * m * (k > 256 ? 2 : 1), 0xAB);
    std::vector<uint16_t> o((size_t)n * dim, 0xABAB);
    const float book = 0.0f;
    CHECK(vq_pq_quantize_host(ctx, VQ_EUCLIDEAN, x.data(), n, m, sd, k, &book, rotation ? &book : nullptr,
                              codes ? c.data() : nullptr, out ? o.data() : nullptr) == VQ_OK);
    const float add = rotation ? 1.0f : 0.0f;
    bool same = true;
    for (int64_t i = 0; i < n; ++i)
        for (int s = 0; s < m; ++s) {
            const size_t p = (size_t)i * m + s;
            const uint16_t want = code_of(x[p * sd] + add, k);
            if (codes) same = same && (k > 256 ? ((const uint16_t *)c.data())[p] : c[p]) == want;
            for (int t = 0; out && t < sd; ++t) same = same && o[p * sd + t] == half_of(x[p * sd + t] + add, want);
        }
    CHECK(same);
}

int main() {
    vq_ctx *first = open_ctx(0), *second = open_ctx(1);

    // a context whose device is not the calling thread's current one: the first staged copy makes the
    // streams and events of its pipeline, and they have to be its own device's
    (void)hipSetDevice(0);
    copy_there_and_back(second, (17u << 20) + 5);
    CHECK(second->up && second->up->device == 1 && second->down->device == 1 && second->pipe_up[0]->device == 1);
    (void)hipSetDevice(0);
    batch(second, 30000, 16, 8, 200, false, true, true);
    std::thread other([&] {  // a thread's current device is 0 at its start
        copy_there_and_back(second, (18u << 20) + 77);
    });
    other.join();

    // around the limits of the staged copies and the chunks; above 64 MB with the copying threads
    for (size_t bytes : {(size_t)(4u << 20) - 1, (size_t)(4u << 20), (size_t)(4u << 20) + 1, (size_t)5000003,
                         (size_t)(16u << 20) - 1, (size_t)(16u << 20), (size_t)(16u << 20) + 4097, (size_t)(70u << 20) + 13})
        copy_there_and_back(first, bytes);
    // uploads below 16 MiB and downloads below 4 MiB are the runtime's: one transfer
    for (int mb : {1, 3, 5, 15, 16, 20}) {
        std::vector<uint8_t> h((size_t)mb << 20, 9), d(h.size());
        int n0 = cpu_hip::copies;
        CHECK(vq_h2d(first, d.data(), h.data(), h.size()) == VQ_OK && d == h);
        CHECK((cpu_hip::copies - n0 == 1) == (mb < 16));
        n0 = cpu_hip::copies;
        CHECK(vq_d2h(first, h.data(), d.data(), h.size()) == VQ_OK);
        CHECK((cpu_hip::copies - n0 == 1) == (mb < 4));
    }
    // a large copy is few transfers: the copy engine stands still between two of them
    {
        std::vector<uint8_t> h(130u << 20, 7), d(h.size());
        const int n0 = cpu_hip::copies;
        CHECK(vq_h2d(first, d.data(), h.data(), h.size()) == VQ_OK && d == h);
        CHECK(cpu_hip::copies - n0 <= 9);
    }
    // page-locked memory goes to the copy engine as it is
    void *pin = nullptr;
    CHECK(hipHostMalloc(&pin, 20u << 20, hipHostMallocDefault) == hipSuccess);
    std::vector<uint8_t> dev(20u << 20);
    std::memset(pin, 0x5A, dev.size());
    const int before = cpu_hip::copies;
    CHECK(vq_h2d(first, dev.data(), pin, dev.size()) == VQ_OK && dev == std::vector<uint8_t>(dev.size(), 0x5A));
    CHECK(cpu_hip::copies == before + 1);
    (void)hipHostFree(pin);

    // batches: in place, one chunk, pipelined with and without the copying threads; either output alone
    for (int64_t n : {1, 8, 9, 2048, 2049, 8192, 8193, 33001}) batch(first, n, 16, 8, 256, false, true, true);
    batch(first, 84003, 16, 8, 256, false, true, true);
    batch(first, 33001, 16, 8, 100, false, true, false);
    batch(first, 33001, 16, 8, 100, false, false, true);
    batch(first, 33001, 16, 8, 1000, false, true, true);
    batch(first, 33001, 16, 8, 256, true, true, true);
    batch(first, 5, 1, 2000000, 256, false, true, true);  // a row longer than a chunk
    {
        const int64_t n = 30001;
        const int dim = 96, stages = 4;
        std::vector<float> x((size_t)n * dim);
        for (size_t i = 0; i < x.size(); ++i) x[i] = (float)(i % 777);
        std::vector<uint8_t> c((size_t)n * stages, 0xAB);
        std::vector<uint16_t> o((size_t)n * dim, 0xABAB);
        const float book = 0.0f;
        CHECK(vq_rvq_quantize_host(first, VQ_EUCLIDEAN, x.data(), n, dim, stages, 64, &book, 0.0f, c.data(), o.data()) == VQ_OK);
        bool same = true;
        for (size_t i = 0; i < x.size(); ++i) {
            const uint16_t want = code_of(x[i / (dim / stages) * (dim / stages)], 64);
            same = same && c[i / (dim / stages)] == want && o[i] == half_of(x[i], want);
        }
        CHECK(same);
    }

    // a copy or a computation that fails half way: an error, nothing left running, the context as before
    for (int at : {1, 3, 7}) {
        const std::vector<uint8_t> h = pattern(20u << 20, 1);
        std::vector<uint8_t> d(h.size());
        cpu_hip::copies = 0;
        cpu_hip::fail_copy_at = at;
        CHECK(vq_h2d(first, d.data(), h.data(), h.size()) == VQ_ERR_HIP);
        cpu_hip::copies = 0;
        CHECK(vq_d2h(first, d.data(), const_cast<uint8_t *>(h.data()), h.size()) == VQ_ERR_HIP);
        cpu_hip::fail_copy_at = 0;
        runs = 0;
        fail_run_at = at;
        std::vector<float> x((size_t)58000 * 128, 1.0f);
        std::vector<uint8_t> c((size_t)58000 * 16);
        const float book = 0.0f;
        CHECK(vq_pq_quantize_host(first, VQ_EUCLIDEAN, x.data(), 58000, 16, 8, 256, &book, nullptr, c.data(), nullptr) ==
              VQ_ERR_UNSUPPORTED);
        fail_run_at = 0;
        copy_there_and_back(first, 17u << 20);
        batch(first, 20000, 16, 8, 256, false, true, true);
    }

    // two contexts in two threads at once
    std::thread a([&] { batch(second, 84000, 16, 8, 256, false, true, true); });
    batch(first, 20001, 16, 8, 256, false, true, true);
    a.join();

    close_ctx(first);
    close_ctx(second);
    if (failures) {
        std::fprintf(stderr, "host copies: %d check(s) failed\n", failures);
        return 1;
    }
    std::printf("host copies: ok\n");
    return 0;
}

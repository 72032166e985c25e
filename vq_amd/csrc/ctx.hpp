// Shared host-side state of libvqhip: the context, error reporting, the grow-only device
// workspace and the per-kernel-class event timing.
#pragma once
#include <hip/hip_runtime.h>

#include <cstdarg>
#include <cstdint>
#include <cstdio>
#include <functional>
#include <string>
#include <vector>

#include "../../include/vq_hip.h"

struct DevBuf {
    void *p = nullptr;
    size_t cap = 0;
};

namespace vqh {
class CopyCrew;  // host_batch.hpp
}

struct vq_ctx {
    int device = 0;
    hipStream_t stream = nullptr;
    hipEvent_t ev0 = nullptr, ev1 = nullptr;
    // second stream of the LBG update: the small clusters' gather path runs beside the streaming sums
    hipStream_t side = nullptr;
    hipEvent_t ev_fork = nullptr, ev_join = nullptr;
    std::string err;
    // grow-only device workspace
    DevBuf flags, tables, hist, seg, part_sum, perm, leaf_desc, leaf_sum, codes, idx, reseed, cnorm;
    DevBuf tsvq_sq;              // TSVQ build: squared deviations of a level
    DevBuf tsvq_split;           // TSVQ build: the small per-level tables of the nodes being split
    DevBuf tsvq_level;           // TSVQ build: the level's uploaded tables and the leaf sums of its node means
    DevBuf tsvq_means;           // TSVQ build: the means of all nodes, read back once at the end
    DevBuf tsvq_scan;            // TSVQ build: workspace of the partition's prefix scan
    DevBuf tsvq_km;              // TSVQ build with 2-means splits: centroids, part sums, flags, draws of a level
    void *lbg_pin = nullptr;     // LBG: page-locked index streams and results of a fit
    size_t lbg_pin_cap = 0;
    void *tsvq_pin = nullptr;    // TSVQ build: page-locked staging of a level's tables and decisions
    size_t tsvq_pin_cap = 0;
    // host rows on their way through the GPU (host_batch.hpp): page-locked and device slots of the chunks
    // in flight, the streams and events that order them, the threads that copy.  Held until the context is
    // closed; four chunks and their results, so bounded: 64 MiB for copies, 25 MB for product quantizers and
    // trees, 100 MB for residual quantizers (rows longer than a chunk: four rows)
    static constexpr int kPipe = 4;
    void *pipe_pin = nullptr;
    size_t pipe_pin_cap = 0;
    DevBuf pipe_dev, pipe_rot;
    hipStream_t up = nullptr, down = nullptr;
    hipEvent_t pipe_up[kPipe] = {}, pipe_run[kPipe] = {}, pipe_down[kPipe] = {};
    vqh::CopyCrew *crew = nullptr;
    DevBuf tsvq_gsum, tsvq_guess, tsvq_maps;  // per group of 32 squares: sum, binade guess, integer maps
    DevBuf tsvq_bsum, tsvq_segmaps;           // per block of groups: f64 sum; per run of groups: composed map
    int tsvq_var_path = 0;       // 0 = composed integer maps, 1 = one chain of adds per column
    DevBuf pad_x, pad_cb;        // rows and codebooks whose column blocks are padded to a multiple of 8 floats
    bool pad_held = false;       // pad_x holds rows that a call still reads: nothing pads into it meanwhile
    DevBuf pad_rows;             // the same for a fit of more than 256 centroids, whose passes may pad slices of their own
    DevBuf mfma_tab, mfma_list, mfma_stat;  // tables, re-check list and counters of the matrix-core assignment
    int mfma_stat_cur = 0;       // which of the two sets of counters in mfma_stat the last pass used
    int recheck_src = 0;         // where the last pass counted its undecided pairs: 1 mfma_stat, 2 mfma_list, 3 the fixed scratch
    int assign_path = 0;         // 0 = matrix cores where a kernel exists, 1 = vector ALU only
    int few_path = 0;            // 0 = a few rows in one launch, 1 = by the kernels of longer calls
    // while an encode goes through stages that each have their own centroids: the operand tables of all of
    // them are made in one launch, at the first (launch_mfma_wide)
    struct StageTables {
        const float *cb = nullptr;  // [stages][k][dim]
        int stages = 0, stage = 0;
        bool ready = false;
    } stage_tables;
    bool lbg_small_lds_set = false;  // dynamic-LDS limit granted to k_lbg_update_small
    int compute_units = 0;       // of the context's GPU (0: not asked for yet)
    uint32_t decode_flat_set = 0;  // the kernels of launch_decode_any whose dynamic-LDS limit is granted, a bit each
    int decode_lds_set[4] = {0, 0, 0, 0};  // dynamic-LDS limit already granted to the four resident decode kernels
    uint64_t quad_lds_set[2] = {0, 0};  // dynamic-LDS limit granted to k_tsvq_descend_quad without and with its output, a bit per instance
    int tsvq_descend_path = 0;   // 0 = one inner product per node where it decides (cosine, L2), 1 = two distances per node always
    int procrustes_path = 0;     // 0 = Newton-Schulz polar factor first, SVD when it does not converge; 1 = SVD only
    // vq_assign_noalloc: the device address of this GPU's file-scope scratch array, and whether a
    // call that must not allocate is running (then `ensure` refuses to grow the workspace)
    unsigned char *static_scratch = nullptr;
    bool no_alloc = false;
    DevBuf tmp_a, tmp_b, tmp_c, tmp_d, tmp_e, tmp_f;  // scratch of the RVQ / OPQ / TSVQ entry points
    // codebooks above 256 centroids: chunk tables, chunk winners, running minimum, merged codes,
    // the LBG's assignment, sort keys in and out, the sort's workspace, per-cluster tables, flags
    DevBuf big_chunk, big_win, big_wind, big_best, big_fresh, big_codes, big_keys, big_sorted, big_sort_tmp, big_tables,
        big_flags;
    // optional per-kernel-class timing (HIP events on the stream)
    bool prof_on = false;
    std::vector<hipEvent_t> prof_pool;
    struct Span {
        int cls;
        hipEvent_t a, b;
        bool own_a = true, own_b = true;  // false: the event belongs to another span (returned to the pool once)
    };
    std::vector<Span> prof_open;
    double prof_ms[VQ_PROF_CLASSES] = {0};
    int64_t prof_launches[VQ_PROF_CLASSES] = {0};
};

namespace vqh {

std::string &create_error();

inline int32_t fail(vq_ctx *ctx, int32_t code, const char *fmt, ...) {
    char buf[512];
    va_list ap;
    va_start(ap, fmt);
    vsnprintf(buf, sizeof buf, fmt, ap);
    va_end(ap);
    if (ctx)
        ctx->err = buf;
    else
        create_error() = buf;
    return code;
}

#define VQ_HIP(ctx, call)                                                                          \
    do {                                                                                           \
        hipError_t e__ = (call);                                                                   \
        if (e__ != hipSuccess) {                                                                   \
            (void)hipGetLastError(); /* the runtime keeps the error until it is read: a later   */ \
                                     /* check of a good launch would report this one again      */ \
            return vqh::fail(ctx, e__ == hipErrorOutOfMemory ? VQ_ERR_OOM : VQ_ERR_HIP,            \
                             "%s: %s (%s:%d)", #call, hipGetErrorString(e__), __FILE__, __LINE__); \
        }                                                                                          \
    } while (0)

#define VQ_TRY(expr)                    \
    do {                                \
        int32_t rc__ = (expr);          \
        if (rc__ != VQ_OK) return rc__; \
    } while (0)

inline int32_t ensure(vq_ctx *ctx, DevBuf &b, size_t bytes) {
    if (bytes <= b.cap) return VQ_OK;
    if (ctx->no_alloc)
        return fail(ctx, VQ_ERR_UNSUPPORTED, "this shape needs a workspace allocation, which this entry point may not make");
    if (b.p) {
        VQ_HIP(ctx, hipStreamSynchronize(ctx->stream));
        VQ_HIP(ctx, hipFree(b.p));
        b.p = nullptr;
        b.cap = 0;
    }
    size_t want = bytes + bytes / 8 + 256;
    VQ_HIP(ctx, hipMalloc(&b.p, want));
    b.cap = want;
    return VQ_OK;
}

// Gives a workspace buffer back once nothing on the context's streams uses it.
inline int32_t release(vq_ctx *ctx, DevBuf &b) {
    if (!b.p) return VQ_OK;
    VQ_HIP(ctx, hipStreamSynchronize(ctx->stream));
    if (ctx->side) VQ_HIP(ctx, hipStreamSynchronize(ctx->side));
    VQ_HIP(ctx, hipFree(b.p));
    b = DevBuf();
    return VQ_OK;
}

// Page-locked host memory of the context, grow-only (the device reads and writes it in place).
inline int32_t ensure_pinned(vq_ctx *ctx, void *&p, size_t &cap, size_t bytes) {
    if (bytes <= cap) return VQ_OK;
    if (p) {
        VQ_HIP(ctx, hipStreamSynchronize(ctx->stream));
        VQ_HIP(ctx, hipHostFree(p));
        p = nullptr;
        cap = 0;
    }
    const size_t want = bytes + bytes / 8 + 4096;
    VQ_HIP(ctx, hipHostMalloc(&p, want, hipHostMallocDefault));
    cap = want;
    return VQ_OK;
}

inline unsigned cdiv(int64_t a, int64_t b) { return (unsigned)((a + b - 1) / b); }

inline hipEvent_t prof_event(vq_ctx *ctx) {
    if (!ctx->prof_pool.empty()) {
        hipEvent_t e = ctx->prof_pool.back();
        ctx->prof_pool.pop_back();
        return e;
    }
    hipEvent_t e = nullptr;
    (void)hipEventCreate(&e);
    return e;
}

struct ProfSpan {
    vq_ctx *ctx;
    int cls;
    hipEvent_t a = nullptr;
    ProfSpan(vq_ctx *c, int k) : ctx(c), cls(k) {  // k < 0: no span
        if (ctx->prof_on && k >= 0) {
            a = prof_event(ctx);
            (void)hipEventRecord(a, ctx->stream);
        }
    }
    ~ProfSpan() {
        if (a) {
            hipEvent_t b = prof_event(ctx);
            (void)hipEventRecord(b, ctx->stream);
            ctx->prof_open.push_back({cls, a, b, true, true});
        }
    }
};

// Resolves the recorded spans; the stream must have been synchronised.
inline void prof_collect(vq_ctx *ctx) {
    for (auto &sp : ctx->prof_open) {
        float ms = 0.f;
        if (hipEventElapsedTime(&ms, sp.a, sp.b) == hipSuccess) {
            ctx->prof_ms[sp.cls] += ms;
            ctx->prof_launches[sp.cls] += 1;
        }
    }
    for (auto &sp : ctx->prof_open) {
        if (sp.own_a) ctx->prof_pool.push_back(sp.a);
        if (sp.own_b) ctx->prof_pool.push_back(sp.b);
    }
    ctx->prof_open.clear();
}

// Argument checks shared by the entry points that take a row matrix and codebooks.
// k_max: 256 where the codes are bytes, 65536 where they are 16 bits wide.
int32_t check_common(vq_ctx *ctx, const void *x, int64_t n, int64_t ld, int32_t m, int32_t sd, int32_t k,
                     int32_t k_max = 256);

// Launchers defined in vq_api.hip, used by the RVQ / OPQ entry points.
// d_dist (optional, n x m floats): receives the chosen centroids' distances where the kernel that runs
// computes them anyway; *dist_written says whether it did.
// d_out16 (optional, n x m * sd binary16 values, 16-byte aligned): receives the chosen centroids themselves
// where the kernel that runs has them at hand; *out_written says whether it did.
// pend (optional; one column block, and only where assign_pending_fusable says so): a residual
// update that the pass applies to the rows before it scores them, d_x[i] = src[i] - cb[codes[i]]
// with src = the rows of d_x themselves (src null: d_x is updated in place) or other rows of stride
// src_ld that stay as they are.
struct PendingUpdate {
    const float *cb;
    const uint8_t *codes;
    const float *src;
    int64_t src_ld;
};
int32_t assign_codes(vq_ctx *ctx, int32_t metric, const float *d_x, int64_t n, int64_t ld, int32_t m,
                     int32_t sd, int32_t k, const float *d_codebooks, uint8_t *d_codes, float *d_dist = nullptr,
                     bool *dist_written = nullptr, const PendingUpdate *pend = nullptr, uint16_t *d_out16 = nullptr,
                     bool *out_written = nullptr);
// Up to this many (row, column block) pairs an assignment runs as one workgroup per pair, one launch
// (k_assign_few): two rounds of workgroups; the matrix-core kernels take two to four launches.  The faster way
// at every width, k and metric up to there, and the longer the codebook the more, although each workgroup
// reads all of it.  32 rows of 16 blocks of 8 floats, k = 256, Euclidean: 4.1 us against 6.3;
// 512 rows of one block of 128 floats, k = 256 10 and 20, 1024 floats, k = 256 59 and 78 (256 rows: 32 and 79),
// k = 1024 227 and 1220; Manhattan, 1024 floats, k = 256: 59 and 217; a residual encode of 512 x 1024, four
// stages: 232 and 426.
constexpr int64_t kFewPairs = 512;
constexpr int32_t kFewWidth = 1280;  // the widest block that the kernels of longer calls take, whatever the number of rows
template <typename CodeT>
int32_t assign_few(vq_ctx *ctx, int32_t metric, const float *d_x, int64_t n, int64_t ld, int32_t m, int32_t sd, int32_t k,
                   const float *d_codebooks, CodeT *d_codes, uint16_t *d_out16);
inline bool assign_few_applicable(const vq_ctx *ctx, int64_t n, int32_t m, int32_t sd) {
    return ctx->assign_path == 0 && ctx->few_path == 0 && n * m <= kFewPairs && sd <= kFewWidth;
}
// Whether the assignment of these rows (one column block of sd floats) runs on the pass that can
// take a pending update along.
bool assign_pending_fusable(const vq_ctx *ctx, int32_t metric, const float *d_x, int64_t n, int64_t ld, int32_t sd,
                            int32_t k, const float *d_codebook);

// Sets ctx->compute_units.  (The runtime's query is 0.3 us, a tenth of a small call.)
int32_t know_compute_units(vq_ctx *ctx);

// The width to which an encode pads the column blocks of such rows (0: not at all), and the copy itself:
// n rows of m blocks of sd floats to m blocks of sdp floats, zeros after each block.
int encode_pad_width(const vq_ctx *ctx, int32_t metric, const float *d_x, int64_t n, int64_t ld, int32_t m, int32_t sd,
                     int32_t k, const float *d_codebooks);
void pad_blocks(vq_ctx *ctx, const float *d_x, int64_t n, int64_t ld, int32_t m, int32_t sd, int32_t sdp, float *d_y);
// ... and back: n rows of sd floats from rows of sdp.
void unpad_rows(vq_ctx *ctx, const float *d_y, int64_t n, int32_t sd, int32_t sdp, float *d_x);
constexpr size_t kPadKeep = 2u << 30;  // bytes that the context keeps of a padded copy of a call's rows
// Turns to the other set of counters of undecided pairs: this pass's (cleared by the pass before), and the
// next pass's, which this pass clears.
int32_t next_counters(vq_ctx *ctx, uint32_t **now, uint32_t **next);
constexpr int64_t kPadSlice = 96 << 20;  // bytes of padded rows that an encode makes at a time

// Defined in vq_api_host.hip: ends the copying threads.
void drop_crew(vq_ctx *ctx);

// Defined in vq_api_bigk.hip: the same for any k up to 65536 with 16-bit codes, and the LBG above
// 256 centroids (arguments as vq_lbg_fit, already validated).  last: enqueues what follows the last update; the stream has
// been waited for when the call returns.
int32_t assign_codes_u16(vq_ctx *ctx, int32_t metric, const float *d_x, int64_t n, int64_t ld, int32_t m,
                         int32_t sd, int32_t k, const float *d_codebooks, uint16_t *d_codes,
                         uint16_t *d_out16 = nullptr, bool *out_written = nullptr);
int32_t lbg_fit_big(vq_ctx *ctx, const float *d_x, int64_t n, int64_t ld, int32_t m, int32_t sd, int32_t k,
                    int32_t max_iters, const uint32_t *h_init_idx, const uint32_t *h_reseed_stream,
                    int32_t n_reseed, float *d_codebooks, int32_t *h_iters_run, int32_t *h_reseeds_used,
                    const std::function<void()> &last = {});

}  // namespace vqh

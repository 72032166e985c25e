// libvqhip — host side of the C ABI declared in include/vq_hip.h.
// Compile with: hipcc --offload-arch=gfx950 -O3 -ffp-contract=off
//               -Xclang -target-feature -Xclang -packed-fp32-ops
#include <hip/hip_runtime.h>
#include <hip/hip_ext.h>
#include <hip/hip_fp16.h>

#include <algorithm>
#include <cstdarg>
#include <type_traits>
#include <cstdio>
#include <cstring>
#include <string>
#include <mutex>
#include <vector>

#include "ctx.hpp"
#include "assign_exact.hpp"
#include "assign_mfma.hpp"
#include "assign_mfma_lds.hpp"
#include "decode.hpp"
#include "resident_rules.hpp"

#ifndef VQ_MFMA_RUN
#define VQ_MFMA_RUN 8    // tiles of 32 rows per wave in the matrix-core assignment (a power of two)
#endif
#ifndef VQ_MFMA_WGS
#define VQ_MFMA_WGS 3072 // workgroups of the matrix-core assignment: four rounds of three per compute unit
#endif
#ifndef VQ_MFMA_ROUND
#define VQ_MFMA_ROUND 768  // workgroups of one round: three per compute unit
#endif
#ifndef VQ_MFMA_OWN
#define VQ_MFMA_OWN 16  // most tiles per workgroup of a one-round grid
#endif
#include "lbg_update.hpp"
#include "calibrate.hpp"

namespace vqh {
std::string &create_error() {
    thread_local std::string e;
    return e;
}
}  // namespace vqh

using namespace vqh;

static bool lbg_small(int64_t n, int m, int sd, int k, bool residual);

namespace {

// ---- the scratch of vq_assign_noalloc --------------------------------------------------------
// One array per GPU, held from the moment the library is loaded on that GPU until the process
// ends.  Host code never uses the array's name as an address: vq_ctx_create asks the runtime for
// the device address once per context (hipGetSymbolAddress, with the context's device current)
// and everything else goes through that pointer.
constexpr size_t kNoAllocTabBytes = 1u << 20;       // A operands: 64 bytes per (column block, padded centroid)
constexpr int kNoAllocMaxCells = 16384;             // column blocks x centroids (padded to 64) the tables hold
constexpr int kNoAllocMaxM = 1024;
constexpr size_t kNoAllocAuxOff = kNoAllocTabBytes;                                   // aux [m][kMfma8Aux]
constexpr size_t kNoAllocStatOff = kNoAllocAuxOff + vq::kMfma8Aux * sizeof(float) * kNoAllocMaxM + 256;  // counters
constexpr size_t kNoAllocNormOff = kNoAllocStatOff + sizeof(uint32_t) * vq::kStatSlots * vq::kStatStride;
constexpr size_t kNoAllocBytes = kNoAllocNormOff + sizeof(float) * kNoAllocMaxCells;  // centroid norms (cosine)
static_assert(kNoAllocStatOff % 256 == 0 && kNoAllocNormOff % 256 == 0, "scratch areas stay 256-byte aligned");
static __device__ __align__(256) unsigned char scratch[kNoAllocBytes];
// The context whose calls used a GPU's array last (null: none yet).  Another context may take the
// array over once everything on that context's stream has finished; until then its calls are
// refused, because their kernels would overwrite tables that kernels in flight still read.
constexpr int kMaxDevices = 64;
std::mutex g_scratch_mutex;
vq_ctx *g_scratch_owner[kMaxDevices];

// ---- assignment dispatch -------------------------------------------------------------------

template <int METRIC, bool LBG>
int32_t launch_wide_exact(vq_ctx *ctx, const vq::AssignArgs &a, int sd, const uint32_t *list,
                          const uint32_t *count, const uint2 *pairs = nullptr, const uint32_t *pair_count = nullptr);

template <int SD, int G, int METRIC, bool LBG, bool PAD, bool DIST = false>
int32_t launch_static(vq_ctx *ctx, const vq::AssignArgs &a, int sd) {
    if constexpr (!LBG && !DIST && (METRIC == vq::M_L1 || SD <= 6)) {  // (assign_codes asks for no others)
        if (a.dist) return launch_static<SD, G, METRIC, LBG, PAD, true>(ctx, a, sd);
    }
    size_t lds = (size_t)G * a.k * SD * sizeof(float);
    if (METRIC == vq::M_COS) lds += (size_t)G * a.k * sizeof(float);
    auto kern = vq::k_assign_static<SD, G, METRIC, LBG, PAD, DIST>;
    if (lds > 48 * 1024)
        VQ_HIP(ctx, hipFuncSetAttribute(reinterpret_cast<const void *>(kern),
                                        hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
    int64_t tiles = (a.n + 255) / 256;
    int64_t blocks = tiles * (a.m / G);
    if (blocks > 0x7fffffffLL) return fail(ctx, VQ_ERR_UNSUPPORTED, "grid too large");
    {
        ProfSpan sp(ctx, VQ_PROF_ASSIGN_KERNEL);
        hipLaunchKernelGGL(kern, dim3((unsigned)blocks), dim3(256), lds, ctx->stream, a, sd);
    }
    VQ_HIP(ctx, hipGetLastError());
    return VQ_OK;
}

template <int SD, int METRIC, bool LBG, bool PAD = false>
int32_t launch_static_g(vq_ctx *ctx, const vq::AssignArgs &a, int sd = SD) {
    // G column blocks per lane: as many as keep the lane's floats within 32 registers and the codebooks within 64 KB of LDS,
    // where that leaves a workgroup per compute unit: a lane takes its blocks one after the
    // other (6000 x 16 blocks of four, k = 256, Manhattan 44 -> 12.5 us, x 4 of seven, k = 33 13.5 -> 5; but 20,000 x 16 of five, k = 4 9 -> 4.6).
    size_t per = (size_t)a.k * SD * sizeof(float) + (METRIC == vq::M_COS ? a.k * sizeof(float) : 0);
    auto fills = [&](int G) { return (a.n + 255) / 256 * (a.m / G) >= 256; };
    if constexpr (SD * 4 <= 32) {
        if (a.m % 4 == 0 && 4 * per <= 64 * 1024 && fills(4)) return launch_static<SD, 4, METRIC, LBG, PAD>(ctx, a, sd);
    }
    if constexpr (SD * 2 <= 32) {
        if (a.m % 2 == 0 && 2 * per <= 64 * 1024 && fills(2)) return launch_static<SD, 2, METRIC, LBG, PAD>(ctx, a, sd);
    }
    return launch_static<SD, 1, METRIC, LBG, PAD>(ctx, a, sd);
}

// The register width that k_assign_static holds blocks of sd floats in (0: it does not take them): their own, or
// the next of a few widths, whose last floats are zeros.  (256 centroids of 48 floats are 48 KB of LDS.)
int static_width(int sd) {
    return sd <= 6 ? sd : sd <= 8 ? 8 : sd <= 12 ? 12 : sd <= 16 ? 16 : sd <= 24 ? 24 : sd <= 32 ? 32 : sd <= 48 ? 48 : 0;
}

// Whether blocks of 24 floats and more (but 32) go to k_assign_wide_exact instead of k_assign_static: its waves share a
// row's centroids, while a lane takes them one after the other, however few rows there are.  The model is within
// 25 % at 600 to 150,000 rows, 1 to 16 blocks, Manhattan; microseconds, waves / lanes: 24 floats, k = 256, 600 x 4 12 / 41, 6000 x 16 55 / 42, k = 60 600 x 4
// 12 / 11; 40 floats, k = 256, 600 x 4 16 / 70, 20,000 x 4 79 / 77, k = 100, 2000 x 4 16 / 32; 33 floats, k = 256, 2000 x 4 29 / 69, x 16 117 / 71
// (whole pieces are read as such; of other widths a component at a time, and a codebook of more than 32 KB from beyond the
// vector cache).
bool wide_pays(int64_t n, int m, int sd, int k, bool vec) {
    const int w = static_width(sd);
    if (sd < 24 || sd == 32 || w == 0) return false;
    const double pairs = (double)n * m, start = vec ? 7 + 0.2 * sd : 11 + 0.25 * sd;
    const double lanes = (0.19 * w - 2.2 + k * (0.0043 * w + 0.04)) * std::max(1.0, pairs / 120e3);
    const double step = vec ? 8.5e-8 : k * sd > 8192 ? 3.6e-7 : 1.2e-7;
    const double waves = std::max({start, (7 + 0.2 * sd) * (0.35 + pairs / 22e3), 0.5 * start + pairs * k * sd * step});
    return waves < lanes;
}

// The register width that an assignment by k_assign_static takes; 0: k_assign_wide_exact.
int exact_width(const vq::AssignArgs &a, int sd) {
    return wide_pays(a.n, a.m, sd, a.k, sd % 4 == 0 && (reinterpret_cast<uintptr_t>(a.cb) & 15) == 0) ? 0 : static_width(sd);
}

template <int METRIC, bool LBG>
int32_t launch_assign_m(vq_ctx *ctx, const vq::AssignArgs &a, int sd) {
    const bool pad = static_width(sd) != sd;
    switch (exact_width(a, sd)) {
    case 1: return launch_static_g<1, METRIC, LBG>(ctx, a);
    case 2: return launch_static_g<2, METRIC, LBG>(ctx, a);
    case 3: return launch_static_g<3, METRIC, LBG>(ctx, a);
    case 4: return launch_static_g<4, METRIC, LBG>(ctx, a);
    case 5: return launch_static_g<5, METRIC, LBG>(ctx, a);
    case 6: return launch_static_g<6, METRIC, LBG>(ctx, a);
#define PADDED(W) \
    case W: return pad ? launch_static_g<W, METRIC, LBG, true>(ctx, a, sd) : launch_static_g<W, METRIC, LBG>(ctx, a)
    PADDED(8);
    PADDED(12);
    PADDED(16);
    PADDED(24);
    PADDED(32);
    PADDED(48);
#undef PADDED
    default: break;
    }
    if (a.m > 65535) return fail(ctx, VQ_ERR_UNSUPPORTED, "m too large for the generic kernel");
    ProfSpan sp(ctx, VQ_PROF_ASSIGN_KERNEL);
    return launch_wide_exact<METRIC, LBG>(ctx, a, sd, nullptr, nullptr);
}

// 8-float column blocks: bf16-split scores on the matrix cores, undecided rows resolved in the
// same kernel by the reference-order argmin (assign_mfma.hpp).
// Where the tables of k_assign_mfma8 live in the workspace.
struct MfmaTabPtrs {
    vq::u32x4 *atab;
    float *aux;
    uint32_t *stat, *stat_next;  // the counters of this pass; of the next one
    int nb;
};
// The counters of undecided pairs, of the present pass and of the next.
int32_t counters(vq_ctx *ctx, uint32_t **now, uint32_t **next) {
    const size_t n_stat = (size_t)vq::kStatSlots * vq::kStatStride;
    if (!ctx->mfma_stat.p) {
        VQ_TRY(ensure(ctx, ctx->mfma_stat, sizeof(uint32_t) * 2 * n_stat));
        VQ_HIP(ctx, hipMemsetAsync(ctx->mfma_stat.p, 0, sizeof(uint32_t) * 2 * n_stat, ctx->stream));
    }
    *now = (uint32_t *)ctx->mfma_stat.p + ctx->mfma_stat_cur * n_stat;
    *next = (uint32_t *)ctx->mfma_stat.p + (ctx->mfma_stat_cur ^ 1) * n_stat;
    return VQ_OK;
}
int32_t mfma_tab_ptrs(vq_ctx *ctx, int m, int k, MfmaTabPtrs &t) {
    t.nb = 2 * ((k + 63) / 64);  // blocks of 32 centroids, an even number (the kernel scores them in pairs)
    // A operands: 64 lanes x 16 bytes per (s, block of 32 centroids)
    const size_t n_atab = (size_t)m * t.nb * 256;
    if (ctx->no_alloc) {  // the fixed scratch array; vq_assign_noalloc has checked that the shape fits
        t.atab = (vq::u32x4 *)ctx->static_scratch;
        t.aux = (float *)(ctx->static_scratch + kNoAllocAuxOff);
        t.stat = t.stat_next = (uint32_t *)(ctx->static_scratch + kNoAllocStatOff);
        return VQ_OK;
    }
    VQ_TRY(ensure(ctx, ctx->mfma_tab, sizeof(float) * (n_atab + vq::kMfma8Aux * (size_t)m) + 64));
    VQ_TRY(counters(ctx, &t.stat, &t.stat_next));
    float *atab = (float *)ctx->mfma_tab.p;
    t.atab = (vq::u32x4 *)atab;
    t.aux = atab + n_atab;
    return VQ_OK;
}

// tables_ready: the caller's last kernel has already written the tables of these centroids.
// Events ride on the kernel's own dispatch (hipExtLaunchKernelGGL) instead of being recorded
// around it: a record is a packet of its own on the queue and delays the next kernel by several
// microseconds.  With timing on, the kernel's start and stop events are a span of the kernel
// class; started / done (if asked for) receive events that mark the kernel's start and end —
// done is what another stream waits for — or stay null when the launch carries none.
template <int METRIC, bool LBG>
int32_t launch_mfma(vq_ctx *ctx, const vq::AssignArgs &a, bool tables_ready, hipEvent_t *started = nullptr,
                    hipEvent_t *done = nullptr) {
    // a workgroup = 4 column blocks of 8 floats (one 128-byte line per row) against one run of row
    // tiles, or, where m is not a multiple of 4, one column block against four runs
    const int nb = 2 * ((a.k + 63) / 64);
    const bool grouped = a.m % 4 == 0, full = nb == 8;
    // A wave loads the operands of its column block once (16 KB + 8 KB) and amortises them over
    // its run: 8 tiles of 32 rows where that still leaves several rounds of workgroups per compute unit.
    const int64_t tiles = cdiv(a.n, 32);
    const int64_t groups = grouped ? a.m / 4 : a.m, per_run = grouped ? 1 : 4;
    int run_tiles = VQ_MFMA_RUN;
    while (run_tiles > 1 && cdiv(tiles, per_run * run_tiles) * groups < 8192) run_tiles >>= 1;
    // Up to VQ_MFMA_OWN tiles for each workgroup of a single round: what counts then is the time of one
    // workgroup, and every wave makes its operands itself (OWN) instead of waiting for the launch that
    // makes the tables.  Four rounds with that launch -> one round, m = 16, k = 256: 1,000 rows 11.4 -> 8.3 us, 10,000
    // 17 -> 14, 50,000 (9 tiles) 32.9 -> 29.4, 100,000 (17) 49.6 -> 49.3, 200,000 (33) 76 -> 82; k = 64, 50,000
    // 24.1 -> 19.7; m = 10, a column block per workgroup: 100,000 (11) 35.5 -> 32.7, 200,000 (21) 56 -> 66.
    const int64_t share = cdiv(tiles * groups, per_run * VQ_MFMA_ROUND);
    const bool own = !tables_ready && !ctx->no_alloc && share <= VQ_MFMA_OWN;
    if (own) run_tiles = (int)share;
    const int64_t runs = cdiv(tiles, per_run * (int64_t)run_tiles);
    // a workgroup walks over several runs with the operands it has loaded once; the grid is a few
    // rounds of the three workgroups a compute unit holds (768: the slowest workgroup sets the
    // time; one workgroup per run: the operands are loaded 15,000 times), a multiple of 8 per group
    int64_t run_stride = std::max<int64_t>(8, (VQ_MFMA_WGS / groups) / 8 * 8);
    run_stride = std::min<int64_t>(run_stride, cdiv(runs, 8) * 8);
    const int64_t blocks = run_stride * groups;
    if (blocks >= (1LL << 31)) return fail(ctx, VQ_ERR_UNSUPPORTED, "n * m too large for one launch");
    if (own) ctx->mfma_stat_cur ^= 1;  // cleared by the pass before
    MfmaTabPtrs t;
    VQ_TRY(mfma_tab_ptrs(ctx, a.m, a.k, t));
    if (!tables_ready && !own)
        hipLaunchKernelGGL(vq::k_mfma8_prep<METRIC == vq::M_COS>, dim3(a.m), dim3(256), 0, ctx->stream, a.cb, a.m, a.k,
                           nb, t.atab, t.aux, t.stat, t.stat_next);
    vq::Mfma8Tables tb{(const vq::u32x4 *)t.atab, t.aux, t.stat, nb, t.stat_next};
    auto pick = [&](auto SGc, auto FULLc) {
        constexpr int SGv = decltype(SGc)::value;
        constexpr bool FULLv = decltype(FULLc)::value;
        return own ? (const void *)vq::k_assign_mfma8<METRIC, LBG, SGv, FULLv, true>
                   : (const void *)vq::k_assign_mfma8<METRIC, LBG, SGv, FULLv, false>;
    };
    using Four = std::integral_constant<int, 4>;
    using One = std::integral_constant<int, 1>;
    const void *kern = grouped ? (full ? pick(Four{}, std::true_type{}) : pick(Four{}, std::false_type{}))
                               : (full ? pick(One{}, std::true_type{}) : pick(One{}, std::false_type{}));
    hipEvent_t ev_a = nullptr, ev_b = nullptr;
    if (ctx->prof_on) {
        ev_a = prof_event(ctx);
        ev_b = prof_event(ctx);
        ctx->prof_open.push_back({VQ_PROF_ASSIGN_KERNEL, ev_a, ev_b, true, true});
    } else if (done) {
        ev_b = ctx->ev_fork;
    }
    vq::AssignArgs aa = a;
    int64_t runs_arg = runs;
    void *args[] = {&aa, &tb, &run_tiles, &runs_arg, &run_stride};
    if (ev_a || ev_b)
        VQ_HIP(ctx, hipExtLaunchKernel(kern, dim3((unsigned)blocks), dim3(256), args, 0, ctx->stream, ev_a, ev_b, 0u));
    else
        VQ_HIP(ctx, hipLaunchKernel(kern, dim3((unsigned)blocks), dim3(256), args, 0, ctx->stream));
    VQ_HIP(ctx, hipGetLastError());
    if (started) *started = ev_a;
    if (done) *done = ev_b;
    ctx->recheck_src = ctx->no_alloc ? 3 : 1;
    return VQ_OK;
}

// Exact assignment for wide column blocks, on a row range (list == nullptr) or on the list of
// undecided pairs of the matrix-core pass.
template <int METRIC, bool LBG>
int32_t launch_wide_exact(vq_ctx *ctx, const vq::AssignArgs &a, int sd, const uint32_t *list,
                          const uint32_t *count, const uint2 *pairs, const uint32_t *pair_count) {
    const bool vec = sd % 4 == 0 && (reinterpret_cast<uintptr_t>(a.cb) & 15) == 0;
    const bool listed = list != nullptr;
    size_t lds = sizeof(float) * 4 * vq::kWideRows * (size_t)sd;
    // a handful of listed pairs: one per workgroup, the row and slices of every centroid in LDS
    if (listed) lds = std::max(lds, sizeof(float) * ((size_t)sd + vq::kPairWgLdsFloats));
    // ... or eight rows of a single column block per workgroup
    if (listed && a.m == 1) lds = std::max(lds, sizeof(float) * ((size_t)vq::kRowsWg * sd + vq::kRowsWgLdsFloats));
    static_assert(sizeof(float) * 4 * vq::kWideRows * kFewWidth == 160 * 1024, "k_assign_few takes the same widths");
    if (lds > 160 * 1024) return fail(ctx, VQ_ERR_UNSUPPORTED, "sub_dim %d too large", sd);
    auto pick = [&](auto L, auto V) {
        constexpr bool LISTED = decltype(L)::value, VEC = decltype(V)::value;
        return reinterpret_cast<const void *>(vq::k_assign_wide_exact<METRIC, LBG, LISTED, VEC>);
    };
    const void *kern = listed ? (vec ? pick(std::true_type{}, std::true_type{}) : pick(std::true_type{}, std::false_type{}))
                              : (vec ? pick(std::false_type{}, std::true_type{}) : pick(std::false_type{}, std::false_type{}));
    if (lds > 48 * 1024)
        VQ_HIP(ctx, hipFuncSetAttribute(kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds));
    const int64_t groups = (a.n + vq::kWideRows - 1) / vq::kWideRows;
    dim3 grid(listed ? 2048u : (unsigned)std::min<int64_t>((groups + 3) / 4, 1 << 20), listed ? 1u : (unsigned)a.m);
    unsigned exact_blocks = grid.x;
    if (pairs) grid.x += 1024u;  // the workgroups of the two-candidate list (they come first in the grid)
    vq::AssignArgs aa = a;
    int sdv = sd;
    void *args[] = {&aa, &sdv, (void *)&list, (void *)&count, (void *)&pairs, (void *)&pair_count, &exact_blocks};
    VQ_HIP(ctx, hipLaunchKernel(kern, grid, dim3(256), args, lds, ctx->stream));
    return VQ_OK;
}

// Wide column blocks (sub_dim a multiple of 8 above 8): chunked contraction on the bf16 matrix
// cores with split operands, undecided pairs listed for the exact kernel.
template <int METRIC, bool LBG>
int32_t launch_mfma_wide(vq_ctx *ctx, const vq::AssignArgs &a, int sd) {
    const int nb = (a.k + 31) / 32, nkc = sd / 8, nsl = (sd + 31) / 32;
    constexpr bool COS = METRIC == vq::M_COS;
    // Stages of an encode: their tables lie one behind the other like those of column blocks and are made by the
    // first one's launches (9.4 us a stage at k = 256, 128 floats); each has its own counts, the last one's in the header.
    auto &stages = ctx->stage_tables;
    const bool staged = !COS && !LBG && a.m == 1 && stages.cb && a.cb == stages.cb + (size_t)stages.stage * a.k * sd;
    const int mt = staged ? stages.stages : a.m, at = staged ? stages.stage : 0;
    // A operands: 2 x 64 lanes x 16 bytes per (s, 16 dimensions, block of 32 centroids)
    const size_t n_atab = (size_t)mt * ((sd + 15) / 16) * nb * 128 * 4, n_c2 = (size_t)mt * nb * 32;  // floats
    VQ_TRY(ensure(ctx, ctx->mfma_tab, sizeof(float) * (n_atab + 2 * n_c2 + (size_t)mt * nb + (size_t)mt * sd + 2 * mt + 2 * (size_t)mt * nsl + 8) + 64));
    // header (two counts), the list for the all-centroid check, the list for the two-candidate check
    const size_t n_pairs = (size_t)a.n * a.m;
    // ... and the candidates of an eighth of the pairs (a list beyond that goes over all centroids)
    const size_t n_head = staged ? 4 * (size_t)mt : 4;
    const size_t mask_cap = n_pairs / 8 + 4096, n_list = n_head + ((n_pairs + 3) & ~(size_t)3) + ((2 * n_pairs + 3) & ~(size_t)3);
    VQ_TRY(ensure(ctx, ctx->mfma_list, sizeof(uint32_t) * (n_list + 8 * mask_cap)));
    float *atab = (float *)ctx->mfma_tab.p;
    float *c2perm = atab + n_atab;
    float *pen = c2perm + n_c2;
    float *maxc2 = pen + n_c2;  // per block of 32 centroids
    float *mu = maxc2 + (((size_t)mt * nb + 3) & ~(size_t)3);  // 16-byte aligned: read as float4
    uint32_t *count = (uint32_t *)ctx->mfma_list.p;
    uint32_t *list = count + n_head;
    uint2 *pairs = (uint2 *)(list + ((n_pairs + 3) & ~(size_t)3));  // 16-byte aligned
    vq::u32x4 *masks = (vq::u32x4 *)(count + n_list);               // likewise
    float2 *norms = (float2 *)(mu + (size_t)mt * sd);  // sd is a multiple of 8: 8-byte aligned
    int *shifted = (int *)(norms + (size_t)mt * nsl);
    float *sigma = (float *)(shifted + mt);
    const bool own_centre = !COS && vq::wide_own_centre(a.k, sd);
    const bool make = !staged || !stages.ready;
    const float *tab_cb = staged ? stages.cb : a.cb;
    if (!COS && !own_centre && make)
        hipLaunchKernelGGL(vq::k_block_centres, dim3(mt, nsl), dim3(256), 0, ctx->stream, tab_cb, a.k, sd, mu, norms);
    // squared L2, Euclidean: see kWideT and kWideRho
    // cosine, in units of |x|, two candidates: the split of an operand twice as long, 2^-22 for the division by
    // the norm, fp32 accumulation (34 per 8 dimensions + 16) * 2^-24 of partial sums up to 4.2 |x|, the
    // reference's own rounding 2 (sub_dim + 6) * 2^-24
    const float u24 = 5.9604644775390625e-08f, split = 3.0f * 1.52587890625e-05f;
    const float kappa = 2.0f * (2.0f * split + (8.0f + 4.2f * (34.0f * nkc + 16.0f) + 2.0f * (sd + 6.0f)) * u24);
    const bool half = !COS && vq::wide_half(sd, nb);
    const float rho = vq::kWideRho, t = half ? vq::kWideHalfT : vq::kWideT;
    const float twice = half ? vq::kWideHalfTwo : vq::kWideTwo;
    // half: 17 additions per instruction, one instruction per 16 dimensions begun, and a rounding per dimension
    const float acc_err = (half ? 10.0f * nkc + 26.0f : 27.0f * nkc + 28.0f) * u24;
    const float cross = half ? acc_err + rho : split + acc_err;
    const float pen_c2 = acc_err + cross / t, pen_dc = 1.0f / (rho * t);
    // (half: dc is at most 2^-11 ||c||)
    const float lift = 1.001f + 8.0f * (pen_c2 + (half ? 2.4e-7f * pen_dc : 0.0f));
    const float rel = 6.103515625e-05f + 2.0f * (sd + 16.0f) * u24;
    const void *prep = half ? own_centre ? (const void *)vq::k_mfma_wide_bf_prep<false, true, true>
                                         : (const void *)vq::k_mfma_wide_bf_prep<false, true>
                            : own_centre ? (const void *)vq::k_mfma_wide_bf_prep<false, false, true>
                                         : (const void *)vq::k_mfma_wide_bf_prep<COS, false>;
    if (make) {
        vq::u32x4 *atab4 = (vq::u32x4 *)atab;
        int m = mt, k = a.k, nbv = nb, sdv = sd, step = staged ? 4 : 0;
        float pc = pen_c2, pd = pen_dc;
        const float *cb = tab_cb, *cnorm = a.cnorm;
        void *args[] = {&cb, &mu, &norms, &shifted, &m, &k, &nbv, &sdv, &atab4, &c2perm, &maxc2, &count, &pen, &pc, &sigma, &pd, &step, &cnorm};
        VQ_HIP(ctx, hipLaunchKernel(prep, dim3(mt, nb), dim3(256), args, 0, ctx->stream));
        if (staged) stages.ready = true;
    }
    if (staged) {  // this stage's
        atab += (size_t)at * ((sd + 15) / 16) * nb * (half ? 64 : 128) * 4;
        c2perm += (size_t)at * nb * 32;
        pen += (size_t)at * nb * 32;
        maxc2 += (size_t)at * nb;
        mu += (size_t)at * sd;
        shifted += at;
        sigma += at;
        count += 4 * (mt - 1 - at);
    }
    vq::MfmaWideBfTables tb{(const vq::u32x4 *)atab, c2perm, pen, maxc2, mu, shifted, sigma, list, count, pairs, masks, (uint32_t)mask_cap, nb, sd,
                            kappa, twice * cross * t, twice * t / rho, lift, rel};
    const size_t res_lds = vq::wide_res_lds(sd, nb);
    const bool resident = half && !a.pend_cb && res_lds <= 160 * 1024 && a.n * a.m >= vq::kWideResMinRows &&
                          a.ld < ((int64_t)1 << 24);  // (32 rows below 2^31 bytes)
    // a workgroup per compute unit, the same number for every column block: where 256 / m rounds down, some
    // units have none, and the kernel is still the faster one (6,000 rows of 96 blocks of 64, 192 workgroups: 104
    // -> 91 us staged -> resident, 127 blocks, 254: 132 -> 100, 4,000 rows of 200 blocks, 200: 140 -> 113; close to
    // kWideResMinRows 1,500 x 96 49 -> 51)
    const int64_t res_groups = std::max<int64_t>(1, 256 / a.m);
    {
        ProfSpan sp(ctx, VQ_PROF_ASSIGN_KERNEL);
#define WIDE(NB)                                                                                             \
    if (COS)                                                                                                 \
        hipLaunchKernelGGL((vq::k_assign_mfma_wide_bf<false, NB, false, true>), dim3(cdiv(a.n, 128), (unsigned)a.m), \
                           dim3(256), 0, ctx->stream, a, tb);                                                \
    else if (half && a.pend_cb)                                                                              \
        hipLaunchKernelGGL((vq::k_assign_mfma_wide_bf<LBG, NB, true, false, true>), dim3(cdiv(a.n, 128), (unsigned)a.m), \
                           dim3(256), 0, ctx->stream, a, tb);                                                \
    else if (resident) {                                                                                     \
        const void *kern = (const void *)vq::k_assign_mfma_wide_res<LBG, NB>;                                \
        if (res_lds > 48 * 1024)                                                                             \
            VQ_HIP(ctx, hipFuncSetAttribute(kern, hipFuncAttributeMaxDynamicSharedMemorySize, (int)res_lds)); \
        hipLaunchKernelGGL((vq::k_assign_mfma_wide_res<LBG, NB>), dim3((unsigned)res_groups, (unsigned)a.m), \
                           dim3(vq::kWideResThreads), res_lds, ctx->stream, a, tb);                          \
    } else if (half)                                                                                         \
        hipLaunchKernelGGL((vq::k_assign_mfma_wide_bf<LBG, NB, false, false, true>), dim3(cdiv(a.n, 128), (unsigned)a.m), \
                           dim3(256), 0, ctx->stream, a, tb);                                                \
    else if (a.pend_cb)                                                                                           \
        hipLaunchKernelGGL((vq::k_assign_mfma_wide_bf<LBG, NB, true>), dim3(cdiv(a.n, 128), (unsigned)a.m),    \
                           dim3(256), 0, ctx->stream, a, tb);                                                \
    else                                                                                                     \
        hipLaunchKernelGGL((vq::k_assign_mfma_wide_bf<LBG, NB>), dim3(cdiv(a.n, 128), (unsigned)a.m), dim3(256), 0, \
                           ctx->stream, a, tb)
        switch (nb) {
        case 1: WIDE(1); break;
        case 2: WIDE(2); break;
        case 3: WIDE(3); break;
        case 4: WIDE(4); break;
        case 5: WIDE(5); break;
        case 6: WIDE(6); break;
        case 7: WIDE(7); break;
        default: WIDE(8); break;
        }
#undef WIDE
    }
    VQ_HIP(ctx, hipGetLastError());
    ctx->recheck_src = 2;
    if constexpr (!COS) {
        if (resident) {
            hipLaunchKernelGGL((vq::k_wide_follow<METRIC, LBG>), dim3(vq::kFollowPairBlocks + vq::kFollowRowBlocks), dim3(256), 0,
                               ctx->stream, a, sd, (const uint32_t *)list, (const uint32_t *)count, (const vq::u32x4 *)masks,
                               (uint32_t)mask_cap, (const uint2 *)pairs);
            VQ_HIP(ctx, hipGetLastError());
            return VQ_OK;
        }
    }
    // undecided pairs with two candidates and the few that need every centroid, in one launch
    return launch_wide_exact<METRIC, LBG>(ctx, a, sd, list, count, (const uint2 *)pairs,
                                          (const uint32_t *)(count + 1));
}

template <int METRIC, bool LBG>
bool mfma_wide_applicable(const vq_ctx *ctx, const vq::AssignArgs &a, int sd) {
    if (ctx->assign_path == 1 || ctx->no_alloc) return false;  // its lists grow with n: not for a fixed scratch
    if (METRIC != vq::M_SQ && METRIC != vq::M_EUCLID && !(METRIC == vq::M_COS && !LBG)) return false;
    if (sd < 16 || sd % 8 != 0 || a.k > 256 || a.m > 65535) return false;
    // float4 row and centroid loads; the rows of a workgroup and the operand table within 32-bit byte offsets
    if (a.ld % 4 != 0 || ((reinterpret_cast<uintptr_t>(a.x) | reinterpret_cast<uintptr_t>(a.cb)) & 15) != 0)
        return false;
    if (a.ld > (1 << 20) || sd > (1 << 16)) return false;
    return (int64_t)a.n * a.m < (1LL << 32);
}

template <int METRIC, bool LBG>
bool mfma_applicable(const vq_ctx *ctx, const vq::AssignArgs &a, int sd) {
    if (ctx->assign_path == 1) return false;
    if (METRIC != vq::M_SQ && METRIC != vq::M_EUCLID && !(METRIC == vq::M_COS && !LBG)) return false;
    if (sd != 8 || (reinterpret_cast<uintptr_t>(a.cb) & 15) != 0) return false;  // float4 centroid loads
    // the kernel addresses the rows of a wave's run (at most 288 of them) with 32-bit offsets
    if (a.ld > (1 << 20) || a.m > (1 << 16)) return false;
    return a.k <= 256;
}

// 16-float column blocks: one pass with the operands in LDS, undecided rows resolved in the same kernel
// (assign_mfma_lds.hpp).  Against the kernel of wider blocks, its tables and its follow-up (an encode, Euclidean): 600,000 x
// 8 blocks, k = 256 369 -> 181 us, 60,000 x 10 61 -> 34, k = 32 33 -> 24, 1,000 x 10 15.4 -> 11; cosine, with sets of eight, 376 -> 201, 64 -> 36.
template <int METRIC, bool LBG>
bool mfma16_applicable(const vq_ctx *ctx, const vq::AssignArgs &a, int sd) {
    if (ctx->assign_path == 1 || ctx->no_alloc || a.pend_cb) return false;
    if (METRIC != vq::M_SQ && METRIC != vq::M_EUCLID && !(METRIC == vq::M_COS && !LBG)) return false;
    // float4 centroid loads; 32 rows within 32-bit byte offsets
    return sd == 16 && (reinterpret_cast<uintptr_t>(a.cb) & 15) == 0 && a.ld <= (1 << 20) && a.m <= 65535 && a.k <= 256;
}
template <int METRIC, bool LBG> int32_t launch_mfma16(vq_ctx *ctx, const vq::AssignArgs &a) {
    vq::LdsArgs args{};
    args.a = a;
    VQ_TRY(next_counters(ctx, &args.stat, &args.stat_next));
    ProfSpan sp(ctx, VQ_PROF_ASSIGN_KERNEL);
    VQ_HIP(ctx, (vq::launch_mfma_lds<METRIC, 16, LBG ? vq::CODES_LBG : vq::CODES_U8>(ctx->stream, args)));
    return VQ_OK;
}

// Microseconds per iteration of a fit of blocks of 8 floats whose sums go by the lists of members, or are streamed
// (k_lbg_stream8).  The lists and their leaves cost by the (row, block) pair, and more with the centroids among which a
// part's rows are spread.  The streaming kernel costs less per pair, but takes more rounds the fewer clusters share a tile of rows (one wave's
// chain over a part), and its clusters of up to 1024 members go by the lists as well, some from averages of 1800 on.  Odd numbers of
// blocks leave lanes idle in both.  The choice by these models costs 0.3 % on average over 234 shapes, 7 % at most (lists / streamed): 250,000 x 12
// k = 4 129 / 256, 16 129 / 157, 40 132 / 134, 112 155 / 125, 256 212 / 162; x 33 k = 6 288 / 317, 10 287 / 266, 40 290 / 205; 1M x 16
// k = 4 575 / 583, 6 572 / 497; 600,000 x 4 k = 64 133 / 122, 128 140 / 118; 500,000 x 5 k = 64 132 / 119, 200 170 / 123, x 8 k = 24
// 167 / 154; 100,000 x 32 k = 48 142 / 133, 96 153 / 160; 87,148 x 32 k = 53 137 / 144; 60,000 x 48 k = 40 132 / 132, 80 143 / 179; 150,000 x 16
// k = 128 133 / 142; 250,000 x 4 k = 56 68 / 105, 256 98 / 122.
double fit8_lists_us(int64_t n, int m, int k) {
    return 33 + (m % 2 ? 6 : 0) + (double)n * m * 1e-6 * (31.5 + 0.09 * k);
}
double fit8_streamed_us(int64_t n, int m, int k) {
    const double members = (double)n / k;  // of an average cluster
    return 80 + (m % 2 ? 6 : 0) + 420.0 / k + (double)n * m * 1e-6 * (13 + 50.0 / k) + std::max(0.0, 0.066 * (1800 - members));
}
// (four blocks to a workgroup: a last group with idle waves from 61,441 rows on only)
bool stream_pays(int64_t n, int m, int k) {
    return (m % 4 == 0 || n > 15 * vq::kPartRows) && fit8_streamed_us(n, m, k) < fit8_lists_us(n, m, k);
}

// The same of a fit of 8 floats by the faster way and of narrower blocks of their own width, for the choice between them
// (three operations per component and centroid beside the bytes; one block per lane where their number is odd).
// Own width / padded, measured: 250,000 x 12 blocks of 3, k = 32 121 / 131, 80 148 / 131; x 33 of 6, k = 4 362 / 288, x 46 of 7 474 / 386;
// 60,000 x 12 of 6, k = 24 57 / 55, 56 74 / 65; 100,000 x 13 of 5, k = 48 80 / 76, 200 139 / 91; 87,148 x 31 of 4, k = 24 118 / 120, 53 135 / 135, 80 145 / 141; x 13
// of 4, k = 40 70 / 80, 128 98 / 92; 150,000 x 12 of 6, k = 24 93 / 97, 53 113 / 103; 500,000 x 12 of 6, k = 40 267 / 175, 100 405 / 170; 1M x 4 of 4,
// k = 64 195 / 138, 200 354 / 155; 60,007 x 25 of 4, k = 40 86 / 98.
double fit8_us(int64_t n, int m, int k) {
    return stream_pays(n, m, k) ? fit8_streamed_us(n, m, k) : fit8_lists_us(n, m, k);
}
double fit_static_us(int64_t n, int m, int sd, int k) {
    const int w = sd == 7 ? 8 : sd;
    const double alone = m % 2 ? std::max(0.0, 8 - 0.08 * k) : 0.0;
    return 28 + (double)n * m * 1e-6 * (22.5 + 1.9 * std::max(0, w - 4) + 0.022 * (3 * w + 1) * k + alone);
}

// The width to pad every column block to so that the matrix-core kernels take the shape (squared L2,
// Euclidean, cosine; 0: they take it as it is, or padding does not pay).  fit: for the passes of a fit,
// which pads its rows once and whose update then streams blocks of 8 as well (residual: of a residual stage).
// k_assign_static does 3 w + 1 vector instructions per row and centroid (cosine: about 2 w + 26; w: its register
// width), the padded kernels about 600 per row and block and half the bytes more to read.  Its own widths: the
// lines below are where the two took the same time at 20,000-600,000 rows, 12 and 25 blocks; one float
// per block leaves most rows to the exact path of the matrix-core kernels: never.  Widths that it holds with zeros
// behind them (150,000 rows, an assignment, microseconds padded / static, 12 blocks, then 11): 7 floats k = 31 58 / 43, 55 / 46, 48
// 55 / 54, 55 / 49, 64 56 / 67, 53 / 58; 10 floats k = 48 86 / 70, 82 / 62, 60 88 / 83, 83 / 74, 80 94 / 111, 88 / 95; 20 floats
// k = 48 166 / 144, 140 / 121, 60 165 / 156, 139 / 148, 80 173 / 200, 149 / 189; 25 floats k = 60 201 / 193, 185 / 181, 80 210 / 255, 194 / 244;
// cosine, 11 blocks: 7 floats k = 31 56 / 53, 48 57 / 67, 15 floats k = 33 83 / 69, 40 85 / 80, 60 85 / 112, 20 floats k = 48 136 / 123, 60
// 135 / 142; 33 floats, k = 48, 400,000 x 1 52 / 64, 150,000 x 4 81 / 92, k = 33 81 / 72; cosine, 15 floats, k = 33, 20,000 x 16 24.5 /
// 30: so the line is a number of centroids, about the same for all of them and for odd numbers of blocks (few rows have it higher: 30,000 x 11
// of 7, k = 48 24 / 16, of 10, k = 60 29 / 23).  The passes of a fit lie no
// further apart, but its update needs fewer launches where the padded blocks make it a small one (12,000 x 12
// blocks of 10, k = 24, six iterations: 241 against 705 us).  Where the update is a small one at both widths (multiples
// of four floats; per iteration own / padded): 431 x 15 blocks of 4, k = 16 12.5 / 14.8, k = 32 12.9 / 14.7, 10,000 x 15 of 4, k = 64 19.6 / 20.1, 256
// 31 / 24; of 12, k = 16 13 / 15.4, 32 15.4 / 15.9, 64 18.9 / 16; of 20, k = 16 16.8 / 23.5, 32 19.3 / 22.8, 64 26 / 22.7; of 28, k = 32 22.5 / 23.5,
// 64 30 / 23.  Widths that neither takes always gain.
int pad_width(const vq_ctx *ctx, int metric, const vq::AssignArgs &a, int sd, bool fit, bool residual = false) {
    if (ctx->assign_path == 1 || ctx->no_alloc || ctx->pad_held || metric < VQ_SQEUCLIDEAN || metric > VQ_COSINE) return 0;
    if (sd == 1 || a.k < 2 || a.k > vq::kMaxK || a.m > 65535) return 0;
    if (mfma_applicable<vq::M_SQ, true>(ctx, a, sd) || mfma16_applicable<vq::M_SQ, true>(ctx, a, sd) ||
        mfma_wide_applicable<vq::M_SQ, true>(ctx, a, sd))
        return 0;
    const int sdp = (sd + 7) / 8 * 8;
    if (sdp == sd && a.ld % 4 == 0 && ((reinterpret_cast<uintptr_t>(a.x) | reinterpret_cast<uintptr_t>(a.cb)) & 15) == 0) return 0;
    // the limits of those kernels
    if ((int64_t)a.m * sdp > (1 << 20) || sdp > (1 << 16) || a.n * a.m >= (1LL << 32)) return 0;
    const int w = static_width(sd);
    // few rows, whose update is one launch at either width: padding adds its own launches and pays by the scores alone
    if (fit && sd <= 28 && a.k < 40 && lbg_small(a.n, a.m, sd, a.k, residual)) return 0;
    if (fit && sd != sdp && lbg_small(a.n, a.m, sdp, a.k, residual)) return sdp;
    if (fit && sd < 8) return fit8_us(a.n, a.m, a.k) < fit_static_us(a.n, a.m, sd, a.k) ? sdp : 0;
    if (fit && w && w != sd && (w <= 16 || w == 32)) return a.k >= (w == 32 ? 36 : 40) || (w <= 16 && a.m % 2 == 0) ? sdp : 0;
    if (w == sd) {
        const int cost = a.k * (metric == VQ_COSINE ? 2 * sd + 26 : 3 * sd + 1);
        if (metric == VQ_COSINE ? cost < (sd < 8 ? 1500 : 3500)
            : sd > 8            ? (fit ? a.k < 40 : cost < 3500)
                                : sd == 2 || cost < 1600 || (a.m % 4 != 0 && (cost - 1600) * (double)(a.n * a.m) < 5e8))
            return 0;
    } else if (w && a.k < (w == 48 ? 40 : w > 16 ? 60 : metric == VQ_COSINE ? (w == 8 ? 32 : 33) : w == 8 ? 48 : 60)) {
        return 0;
    }
    return sdp;
}

void launch_pad(vq_ctx *ctx, const float *x, int64_t n, int64_t ld, int m, int sd, int sdp, float *y) {
    hipLaunchKernelGGL(vq::k_pad_blocks, dim3(cdiv(n * m * (sdp / 4), 1024)), dim3(256), 0, ctx->stream, x, n, ld, m, sd,
                       sdp, y);
}

template <bool LBG>
int32_t launch_assign(vq_ctx *ctx, int metric, const vq::AssignArgs &a, int sd, bool tables_ready = false,
                      hipEvent_t *started = nullptr, hipEvent_t *done = nullptr) {
    if (started) *started = nullptr;
    if (done) *done = nullptr;
    if (metric == VQ_SQEUCLIDEAN && mfma_applicable<vq::M_SQ, LBG>(ctx, a, sd))
        return launch_mfma<vq::M_SQ, LBG>(ctx, a, tables_ready, started, done);
    if (metric == VQ_EUCLIDEAN && mfma_applicable<vq::M_EUCLID, LBG>(ctx, a, sd))
        return launch_mfma<vq::M_EUCLID, LBG>(ctx, a, tables_ready, started, done);
    if constexpr (!LBG)
        if (metric == VQ_COSINE && mfma_applicable<vq::M_COS, false>(ctx, a, sd))
            return launch_mfma<vq::M_COS, false>(ctx, a, tables_ready, started, done);
    if (metric == VQ_SQEUCLIDEAN && mfma16_applicable<vq::M_SQ, LBG>(ctx, a, sd)) return launch_mfma16<vq::M_SQ, LBG>(ctx, a);
    if (metric == VQ_EUCLIDEAN && mfma16_applicable<vq::M_EUCLID, LBG>(ctx, a, sd)) return launch_mfma16<vq::M_EUCLID, LBG>(ctx, a);
    if constexpr (!LBG)
        if (metric == VQ_COSINE && mfma16_applicable<vq::M_COS, false>(ctx, a, sd)) return launch_mfma16<vq::M_COS, false>(ctx, a);
    if constexpr (!LBG)
        if (metric == VQ_COSINE && mfma_wide_applicable<vq::M_COS, false>(ctx, a, sd))
            return launch_mfma_wide<vq::M_COS, false>(ctx, a, sd);
    if (metric == VQ_SQEUCLIDEAN && mfma_wide_applicable<vq::M_SQ, LBG>(ctx, a, sd))
        return launch_mfma_wide<vq::M_SQ, LBG>(ctx, a, sd);
    if (metric == VQ_EUCLIDEAN && mfma_wide_applicable<vq::M_EUCLID, LBG>(ctx, a, sd))
        return launch_mfma_wide<vq::M_EUCLID, LBG>(ctx, a, sd);
    if (metric == VQ_SQEUCLIDEAN) return launch_assign_m<vq::M_SQ, LBG>(ctx, a, sd);
    if constexpr (!LBG) {  // the passes of a fit are squared Euclidean
        if (metric == VQ_EUCLIDEAN) return launch_assign_m<vq::M_EUCLID, false>(ctx, a, sd);
        if (metric == VQ_COSINE) return launch_assign_m<vq::M_COS, false>(ctx, a, sd);
        if (metric == VQ_MANHATTAN) return launch_assign_m<vq::M_L1, false>(ctx, a, sd);
    }
    return fail(ctx, VQ_ERR_UNSUPPORTED, "metric %d has no kernel", metric);
}

// Reconstruction with the codebook table resident in LDS (up to 128 KB, one workgroup of 1024 threads per
// compute unit walking over the output, two where the table leaves room): a thread makes one 16-byte piece of the
// output per step, eight f16 values (F16; sub_dim a multiple of 8) or four f32 values (sub_dim a
// multiple of 4), so a wave's stores are consecutive bytes, its code reads consecutive
// bytes, and the centroid comes from LDS instead of a scattered read of the table through
// the vector cache.  U pieces per thread are in flight.  blockIdx.y: a group of G column blocks, where the table
// of all of them does not fit.  A workgroup takes runs of whole rows, so that a piece's place in its run is
// divided in 32 bits; the stores pass the caches, so runs, and a group's share of a row, have to fill their lines.
// Bound by the stores; decode_resident_blocks has its times and the gather's.
template <bool F16, typename CodeT>
__global__ void __launch_bounds__(1024) k_decode_resident(const CodeT *__restrict__ codes, int64_t n, int m, int sd,
                                                          int k, int G, const float *__restrict__ cb,
                                                          vq::u32x4 *__restrict__ out) {
    extern __shared__ __attribute__((aligned(16))) vq::u32x4 tab[];  // [blocks of the group * k][pieces of a centroid]
    constexpr int U = F16 ? 4 : 8;  // pieces in flight per thread
    const uint32_t pieces = F16 ? sd / 8 : sd / 4;  // 16-byte output pieces per centroid
    const int s0 = (int)blockIdx.y * G, mg = m - s0 < G ? m - s0 : G;
    const uint32_t entries = (uint32_t)mg * k * pieces;
    cb += (size_t)s0 * k * sd;
    for (uint32_t e = threadIdx.x; e < entries; e += 1024) {
        if constexpr (F16) {
            const float4 a = reinterpret_cast<const float4 *>(cb)[2 * (size_t)e];
            const float4 b = reinterpret_cast<const float4 *>(cb)[2 * (size_t)e + 1];
            auto two = [](float lo, float hi) {
                return (uint32_t)__half_as_ushort(__float2half_rn(lo)) | ((uint32_t)__half_as_ushort(__float2half_rn(hi)) << 16);
            };
            tab[e] = vq::u32x4{two(a.x, a.y), two(a.z, a.w), two(b.x, b.y), two(b.z, b.w)};
        } else {
            tab[e] = reinterpret_cast<const vq::u32x4 *>(cb)[e];
        }
    }
    __syncthreads();
    const uint32_t per_row = (uint32_t)mg * pieces;
    // rows of a run: eight at a time, which end with a line whatever m is
    const int64_t rows = U * 1024 / per_row >= 8 ? U * 1024 / per_row / 8 * 8 : U * 1024 / per_row > 1 ? U * 1024 / per_row : 1;
    for (int64_t row0 = blockIdx.x * rows; row0 < n; row0 += gridDim.x * rows) {
        const uint32_t count = (uint32_t)(n - row0 < rows ? n - row0 : rows) * per_row;
        const CodeT *run = codes + row0 * m + s0;
        vq::u32x4 *to = out + (row0 * m + s0) * pieces;
        for (uint32_t l0 = threadIdx.x; l0 < count; l0 += U * 1024) {
            uint32_t code[U], at[U], entry[U];
#pragma unroll
            for (int u = 0; u < U; ++u) {
                const uint32_t l = l0 + 1024u * u < count ? l0 + 1024u * u : l0;
                const uint32_t row = l / per_row, within = l - row * per_row;
                const uint32_t s = pieces == 1 ? within : within / pieces;
                code[u] = run[row * (uint32_t)m + s];
                at[u] = row * (uint32_t)m * pieces + within;
                entry[u] = s * (uint32_t)k * pieces + (within - s * pieces);
            }
            vq::u32x4 v[U];
#pragma unroll
            for (int u = 0; u < U; ++u) v[u] = tab[entry[u] + code[u] * pieces];
#pragma unroll
            for (int u = 0; u < U; ++u)
                if (l0 + 1024u * u < count) __builtin_nontemporal_store(v[u], to + at[u]);
        }
    }
}

__global__ void __launch_bounds__(256) k_copy_f32(const float4 *__restrict__ src,
                                                  float4 *__restrict__ dst, int64_t n4,
                                                  const float *__restrict__ src_tail,
                                                  float *__restrict__ dst_tail, int tail) {
    int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
    int64_t stride = (int64_t)gridDim.x * 256;
    for (; i < n4; i += stride) dst[i] = src[i];
    if (blockIdx.x == 0 && (int)threadIdx.x < tail) dst_tail[threadIdx.x] = src_tail[threadIdx.x];
}

// LDS-resident decode where it is the faster one (decode_resident_blocks).
template <bool F16, typename CodeT>
int32_t launch_decode_resident(vq_ctx *ctx, const CodeT *d_codes, int64_t n, int m, int sd, int k,
                               const float *d_codebooks, void *d_out, bool *done) {
    *done = false;
    const int G = vq::decode_resident_blocks(F16, n, m, sd, k);
    if (G == 0) return VQ_OK;
    const size_t lds = (size_t)k * sd * (F16 ? 2 : 4) * G;
    if ((reinterpret_cast<uintptr_t>(d_codebooks) & 15) || (reinterpret_cast<uintptr_t>(d_out) & 63)) return VQ_OK;
    auto kern = k_decode_resident<F16, CodeT>;
    // the kernel's LDS limit: asked for once per context and kernel
    const int slot = (F16 ? 2 : 0) + (sizeof(CodeT) == 2 ? 1 : 0);
    if ((size_t)ctx->decode_lds_set[slot] < lds) {
        VQ_HIP(ctx, hipFuncSetAttribute(reinterpret_cast<const void *>(kern),
                                        hipFuncAttributeMaxDynamicSharedMemorySize, 128 * 1024));
        ctx->decode_lds_set[slot] = 128 * 1024;
    }
    VQ_TRY(know_compute_units(ctx));
    const int64_t pieces = (int64_t)n * m * (F16 ? sd / 8 : sd / 4);
    const unsigned per_cu = lds <= 64 * 1024 ? 2u : 1u;
    const unsigned groups = cdiv(m, G);
    const unsigned wgs = (unsigned)std::min<int64_t>(std::max<int64_t>(1, (int64_t)ctx->compute_units * per_cu / groups),
                                                     cdiv(pieces, 4096 * groups));
    hipLaunchKernelGGL(kern, dim3(wgs, groups), dim3(1024), lds, ctx->stream, d_codes, n, m, sd, k, G, d_codebooks,
                       (vq::u32x4 *)d_out);
    VQ_HIP(ctx, hipGetLastError());
    *done = true;
    return VQ_OK;
}

// Decode of 8- or 16-bit codes to binary16 bit patterns (F16) or f32.
template <bool F16, typename CodeT>
int32_t decode_codes(vq_ctx *ctx, const CodeT *d_codes, int64_t n, int32_t m, int32_t sd, int32_t k, int32_t k_max,
                     const float *d_codebooks, void *d_out) {
    if (!ctx) return VQ_ERR_INVALID_ARG;
    if (n == 0) return VQ_OK;
    if (!d_codes || !d_codebooks || !d_out || n < 0 || m <= 0 || sd <= 0 || k <= 0 || k > k_max)
        return fail(ctx, VQ_ERR_INVALID_ARG, "Invalid parameter");
    VQ_HIP(ctx, hipSetDevice(ctx->device));
    bool done = false;
    VQ_TRY((launch_decode_resident<F16, CodeT>(ctx, d_codes, n, m, sd, k, d_codebooks, d_out, &done)));
    if (done) return VQ_OK;
    const bool aligned = ((reinterpret_cast<uintptr_t>(d_codebooks) | reinterpret_cast<uintptr_t>(d_out)) & 15) == 0;
    constexpr int piece = F16 ? 8 : 4;
    if (sd % piece == 0 && aligned && (int64_t)m * sd < (1LL << 31))
        hipLaunchKernelGGL((vq::k_decode_gather<F16, CodeT>), dim3(cdiv(n * m * (sd / piece), 1024)), dim3(256), 0,
                           ctx->stream, d_codes, n, m, sd, k, d_codebooks, (vq::u32x4_out *)d_out);
    else {
        VQ_TRY(know_compute_units(ctx));
        VQ_HIP(ctx, (vq::launch_decode_any<F16, CodeT>(ctx->stream, ctx->compute_units, ctx->decode_flat_set, d_codes, n, m, sd, k, d_codebooks,
                                                       d_out)));
    }
    VQ_HIP(ctx, hipGetLastError());
    return VQ_OK;
}

}  // namespace

namespace vqh {
int32_t check_common(vq_ctx *ctx, const void *x, int64_t n, int64_t ld, int32_t m, int32_t sd,
                     int32_t k, int32_t k_max) {
    if (!ctx) return VQ_ERR_INVALID_ARG;
    if (n == 0) return fail(ctx, VQ_ERR_EMPTY_INPUT, "Empty input: at least one vector is required.");
    if (!x || n < 0 || m <= 0 || sd <= 0)
        return fail(ctx, VQ_ERR_INVALID_ARG, "Invalid parameter: null pointer or non-positive size");
    if (ld < (int64_t)m * sd)
        return fail(ctx, VQ_ERR_DIM_MISMATCH, "Dimension mismatch: expected %lld, got %lld",
                    (long long)m * sd, (long long)ld);
    if (k <= 0) return fail(ctx, VQ_ERR_INVALID_ARG, "Invalid parameter: k must be greater than 0");
    if (k > k_max)
        return fail(ctx, VQ_ERR_UNSUPPORTED,
                    k_max <= vq::kMaxK ? "k = %d: the codes of this entry point are uint8, k must be <= 256"
                                       : "k = %d: codes are at most 16 bits wide, k must be <= 65536", k);
    if (n >= (1LL << 32)) return fail(ctx, VQ_ERR_UNSUPPORTED, "n must be below 2^32");
    return VQ_OK;
}


bool assign_pending_fusable(const vq_ctx *ctx, int32_t metric, const float *d_x, int64_t n, int64_t ld, int32_t sd,
                            int32_t k, const float *d_codebook) {
    vq::AssignArgs a;
    a.x = d_x;
    a.n = n;
    a.ld = ld;
    a.m = 1;
    a.k = k;
    a.cb = d_codebook;
    if (k < 1 || sd % 4 != 0) return false;
    return (metric == VQ_SQEUCLIDEAN && mfma_wide_applicable<vq::M_SQ, false>(ctx, a, sd)) ||
           (metric == VQ_EUCLIDEAN && mfma_wide_applicable<vq::M_EUCLID, false>(ctx, a, sd));
}

template <typename CodeT>
int32_t assign_few(vq_ctx *ctx, int32_t metric, const float *d_x, int64_t n, int64_t ld, int32_t m, int32_t sd, int32_t k,
                   const float *d_codebooks, CodeT *d_codes, uint16_t *d_out16) {
    const dim3 grid((unsigned)m, (unsigned)n);
    const size_t lds = sizeof(float) * ((size_t)sd + 4);
#define FEW(M)                                                                                                     \
    hipLaunchKernelGGL((vq::k_assign_few<M, CodeT>), grid, dim3(256), lds, ctx->stream, d_x, ld, m, sd, k, d_codebooks, \
                       d_codes, d_out16)
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
template int32_t assign_few<uint8_t>(vq_ctx *, int32_t, const float *, int64_t, int64_t, int32_t, int32_t, int32_t,
                                     const float *, uint8_t *, uint16_t *);
template int32_t assign_few<uint16_t>(vq_ctx *, int32_t, const float *, int64_t, int64_t, int32_t, int32_t, int32_t,
                                      const float *, uint16_t *, uint16_t *);

int encode_pad_width(const vq_ctx *ctx, int32_t metric, const float *d_x, int64_t n, int64_t ld, int32_t m, int32_t sd,
                     int32_t k, const float *d_codebooks) {
    vq::AssignArgs a{};
    a.x = d_x;
    a.n = n;
    a.ld = ld;
    a.m = m;
    a.k = k;
    a.cb = d_codebooks;
    return pad_width(ctx, metric, a, sd, false);
}

int32_t know_compute_units(vq_ctx *ctx) {
    if (ctx->compute_units == 0) {
        int cus = 0;
        VQ_HIP(ctx, hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, ctx->device));
        ctx->compute_units = cus > 0 ? cus : 1;
    }
    return VQ_OK;
}

void pad_blocks(vq_ctx *ctx, const float *d_x, int64_t n, int64_t ld, int32_t m, int32_t sd, int32_t sdp, float *d_y) {
    launch_pad(ctx, d_x, n, ld, m, sd, sdp, d_y);
}

void unpad_rows(vq_ctx *ctx, const float *d_y, int64_t n, int32_t sd, int32_t sdp, float *d_x) {
    hipLaunchKernelGGL(vq::k_unpad_rows, dim3(cdiv(n * sd, 256)), dim3(256), 0, ctx->stream, d_y, n, sd, sdp, d_x);
}

int32_t next_counters(vq_ctx *ctx, uint32_t **now, uint32_t **next) {
    ctx->mfma_stat_cur ^= 1;
    ctx->recheck_src = 1;
    return counters(ctx, now, next);
}

int32_t assign_codes(vq_ctx *ctx, int32_t metric, const float *d_x, int64_t n, int64_t ld, int32_t m,
                  int32_t sd, int32_t k, const float *d_codebooks, uint8_t *d_codes, float *d_dist,
                  bool *dist_written, const PendingUpdate *pend, uint16_t *d_out16, bool *out_written) {
    if (dist_written) *dist_written = false;
    if (out_written) *out_written = false;
    VQ_TRY(check_common(ctx, d_x, n, ld, m, sd, k));
    if (!d_codebooks || !d_codes) return fail(ctx, VQ_ERR_INVALID_ARG, "Invalid parameter: null pointer");
    if (reinterpret_cast<uintptr_t>(d_codes) & 3)
        return fail(ctx, VQ_ERR_INVALID_ARG, "Invalid parameter: d_codes must be 4-byte aligned");
    if (m > 65535) return fail(ctx, VQ_ERR_UNSUPPORTED, "m must be at most 65535");
    VQ_HIP(ctx, hipSetDevice(ctx->device));
    if (!pend && assign_few_applicable(ctx, n, m, sd)) {
        if (out_written) *out_written = d_out16 != nullptr;
        ProfSpan sp(ctx, VQ_PROF_ENCODE);
        return assign_few<uint8_t>(ctx, metric, d_x, n, ld, m, sd, k, d_codebooks, d_codes, d_out16);
    }
    vq::AssignArgs a;
    a.x = d_x;
    a.n = n;
    a.ld = ld;
    a.m = m;
    a.k = k;
    a.cb = d_codebooks;
    a.cnorm = nullptr;
    a.codes = d_codes;
    a.changed = nullptr;
    a.done = nullptr;
    if (pend) {
        if (m != 1 || !assign_pending_fusable(ctx, metric, d_x, n, ld, sd, k, d_codebooks) || !pend->cb ||
            !pend->codes || (reinterpret_cast<uintptr_t>(pend->cb) & 15) != 0 ||
            (pend->src && (pend->src_ld % 4 != 0 || (reinterpret_cast<uintptr_t>(pend->src) & 15) != 0)))
            return fail(ctx, VQ_ERR_INVALID_ARG, "Invalid parameter: no pass that takes a pending update");
        a.pend_cb = pend->cb;
        a.pend_codes = pend->codes;
        a.pend_src = pend->src;
        a.pend_src_ld = pend->src_ld;
    }
    // the 8-float matrix-core kernel has the chosen centroid's exact distance at hand
    const bool mfma8 = metric != VQ_MANHATTAN && mfma_applicable<vq::M_SQ, false>(ctx, a, sd);
    if (d_dist && dist_written && mfma8) {
        a.dist = d_dist;
        *dist_written = true;
    }
    // ... and the chosen centroid in LDS
    if (d_out16 && out_written && (reinterpret_cast<uintptr_t>(d_out16) & 15) == 0 && mfma8) {
        a.out16 = d_out16;
        *out_written = true;
    }
    ProfSpan sp(ctx, VQ_PROF_ENCODE);
    const int sdp = pend ? 0 : pad_width(ctx, metric, a, sd, false);
    // the kernels for 8 and 16 floats make the norms themselves
    if (metric == VQ_COSINE && !mfma8 && sdp != 8 && sdp != 16 && !mfma16_applicable<vq::M_COS, false>(ctx, a, sd)) {
        float *cnorm = (float *)(ctx->static_scratch + kNoAllocNormOff);
        if (!ctx->no_alloc) {
            VQ_TRY(ensure(ctx, ctx->cnorm, sizeof(float) * (size_t)m * k));
            cnorm = (float *)ctx->cnorm.p;
        }
        hipLaunchKernelGGL(vq::k_centroid_norms, dim3(cdiv((int64_t)m * k, 256)), dim3(256), 0,
                           ctx->stream, d_codebooks, (int64_t)m * k, sd, cnorm);
        a.cnorm = cnorm;
    }
    if (!sdp) {
        // k_assign_static has the distance too: Manhattan, and blocks too narrow for the other kernels (a distance of one
        // component costs the merge less than reading it: 60,000 x 5, k = 600 40 -> 36.7 us)
        if (d_dist && dist_written && !mfma8 && !pend && sd > 1 && (metric == VQ_MANHATTAN ? exact_width(a, sd) != 0 : sd <= 6)) {
            a.dist = d_dist;
            *dist_written = true;
        }
        return launch_assign<false>(ctx, metric, a, sd);
    }
    // padded a slice of rows at a time: the copy is read back from the memory-side cache (256 MB)
    // and the workspace stays small whatever n is
    const int64_t row_bytes = (int64_t)sizeof(float) * m * sdp;
    const int64_t slice = std::min<int64_t>(n, std::max<int64_t>(4096, kPadSlice / row_bytes / 4096 * 4096));
    VQ_TRY(ensure(ctx, ctx->pad_x, (size_t)(slice * row_bytes)));
    VQ_TRY(ensure(ctx, ctx->pad_cb, sizeof(float) * (size_t)m * k * sdp));
    launch_pad(ctx, d_codebooks, (int64_t)m * k, sd, 1, sd, sdp, (float *)ctx->pad_cb.p);
    a.x = (const float *)ctx->pad_x.p;
    a.ld = (int64_t)m * sdp;
    a.cb = (const float *)ctx->pad_cb.p;
    if (d_dist && dist_written && sdp == 8) *dist_written = true;
    for (int64_t r0 = 0; r0 < n; r0 += slice) {
        a.n = std::min(slice, n - r0);
        a.codes = d_codes + r0 * m;
        a.dist = d_dist && sdp == 8 ? d_dist + r0 * m : nullptr;
        launch_pad(ctx, d_x + r0 * ld, a.n, ld, m, sd, sdp, (float *)ctx->pad_x.p);
        VQ_TRY(launch_assign<false>(ctx, metric, a, sdp));
    }
    return VQ_OK;
}

}  // namespace vqh

// =============================================================================================
extern "C" {

int32_t vq_ctx_create(int32_t device, vq_ctx **out) {
    if (!out) return fail(nullptr, VQ_ERR_INVALID_ARG, "out is null");
    *out = nullptr;
    int count = 0;
    hipError_t e = hipGetDeviceCount(&count);
    if (e != hipSuccess || count == 0)
        return fail(nullptr, VQ_ERR_HIP, "no HIP device available (%s)",
                    e == hipSuccess ? "device count is 0" : hipGetErrorString(e));
    if (device < 0 || device >= count)
        return fail(nullptr, VQ_ERR_INVALID_ARG, "device %d out of range [0,%d)", device, count);
    vq_ctx *ctx = new vq_ctx;
    ctx->device = device;
    if ((e = hipSetDevice(device)) != hipSuccess ||
        (e = hipStreamCreate(&ctx->stream)) != hipSuccess ||
        (e = hipEventCreate(&ctx->ev0)) != hipSuccess ||
        (e = hipEventCreate(&ctx->ev1)) != hipSuccess ||
        (e = hipStreamCreate(&ctx->side)) != hipSuccess ||
        (e = hipEventCreate(&ctx->ev_fork)) != hipSuccess ||  // rides on a kernel dispatch as its stop event
        (e = hipEventCreateWithFlags(&ctx->ev_join, hipEventDisableTiming | hipEventReleaseToDevice)) != hipSuccess) {
        int32_t rc = fail(nullptr, VQ_ERR_HIP, "context set-up failed: %s", hipGetErrorString(e));
        delete ctx;
        return rc;
    }
    // this GPU's copy of the scratch array (every GPU holds its own, at its own address)
    void *sp = nullptr;
    if ((e = hipGetSymbolAddress(&sp, HIP_SYMBOL(scratch))) != hipSuccess || !sp) {
        int32_t rc = fail(nullptr, VQ_ERR_HIP, "address of the scratch array: %s", hipGetErrorString(e));
        vq_ctx_destroy(ctx);
        return rc;
    }
    ctx->static_scratch = (unsigned char *)sp;
    *out = ctx;
    return VQ_OK;
}

int32_t vq_ctx_destroy(vq_ctx *ctx) {
    if (!ctx) return VQ_OK;
    (void)hipSetDevice(ctx->device);
    (void)hipStreamSynchronize(ctx->stream);
    if (ctx->side) (void)hipStreamSynchronize(ctx->side);
    DevBuf *bufs[] = {&ctx->flags, &ctx->tables, &ctx->hist, &ctx->perm, &ctx->leaf_desc,
                      &ctx->leaf_sum, &ctx->codes, &ctx->idx, &ctx->reseed, &ctx->cnorm,
                      &ctx->seg, &ctx->part_sum, &ctx->pad_x, &ctx->pad_cb, &ctx->pad_rows, &ctx->pipe_dev, &ctx->pipe_rot, &ctx->mfma_tab, &ctx->mfma_list, &ctx->mfma_stat, &ctx->tsvq_sq, &ctx->tsvq_split, &ctx->tsvq_level, &ctx->tsvq_means, &ctx->tsvq_scan, &ctx->tsvq_km, &ctx->tsvq_bsum, &ctx->tsvq_segmaps, &ctx->tsvq_gsum, &ctx->tsvq_guess, &ctx->tsvq_maps, &ctx->tmp_a, &ctx->tmp_b, &ctx->tmp_c, &ctx->tmp_d, &ctx->tmp_e, &ctx->tmp_f,
                      &ctx->big_chunk, &ctx->big_win, &ctx->big_wind, &ctx->big_best, &ctx->big_fresh, &ctx->big_codes, &ctx->big_keys,
                      &ctx->big_sorted, &ctx->big_sort_tmp, &ctx->big_tables, &ctx->big_flags};
    for (DevBuf *b : bufs)
        if (b->p) (void)hipFree(b->p);
    if (ctx->tsvq_pin) (void)hipHostFree(ctx->tsvq_pin);
    if (ctx->lbg_pin) (void)hipHostFree(ctx->lbg_pin);
    drop_crew(ctx);
    if (ctx->pipe_pin) (void)hipHostFree(ctx->pipe_pin);
    for (int i = 0; i < vq_ctx::kPipe; ++i)
        for (hipEvent_t e : {ctx->pipe_up[i], ctx->pipe_run[i], ctx->pipe_down[i]})
            if (e) (void)hipEventDestroy(e);
    if (ctx->up) (void)hipStreamDestroy(ctx->up);
    if (ctx->down) (void)hipStreamDestroy(ctx->down);
    prof_collect(ctx);
    if (ctx->device >= 0 && ctx->device < kMaxDevices) {
        std::lock_guard<std::mutex> lock(g_scratch_mutex);
        if (g_scratch_owner[ctx->device] == ctx) g_scratch_owner[ctx->device] = nullptr;
    }
    for (hipEvent_t e : ctx->prof_pool) (void)hipEventDestroy(e);
    (void)hipEventDestroy(ctx->ev0);
    (void)hipEventDestroy(ctx->ev1);
    if (ctx->ev_fork) (void)hipEventDestroy(ctx->ev_fork);
    if (ctx->ev_join) (void)hipEventDestroy(ctx->ev_join);
    if (ctx->side) (void)hipStreamDestroy(ctx->side);
    (void)hipStreamDestroy(ctx->stream);
    delete ctx;
    return VQ_OK;
}

const char *vq_last_error(const vq_ctx *ctx) { return ctx ? ctx->err.c_str() : vqh::create_error().c_str(); }

int32_t vq_ctx_sync(vq_ctx *ctx) {
    if (!ctx) return VQ_ERR_INVALID_ARG;
    VQ_HIP(ctx, hipStreamSynchronize(ctx->stream));
    return VQ_OK;
}

void *vq_ctx_stream(vq_ctx *ctx) { return ctx ? (void *)ctx->stream : nullptr; }

int32_t vq_malloc(vq_ctx *ctx, size_t bytes, void **d_ptr) {
    if (!ctx || !d_ptr) return VQ_ERR_INVALID_ARG;
    *d_ptr = nullptr;
    VQ_HIP(ctx, hipSetDevice(ctx->device));
    VQ_HIP(ctx, hipMalloc(d_ptr, bytes ? bytes : 1));
    return VQ_OK;
}

int32_t vq_free(vq_ctx *ctx, void *d_ptr) {
    if (!ctx) return VQ_ERR_INVALID_ARG;
    if (!d_ptr) return VQ_OK;
    VQ_HIP(ctx, hipStreamSynchronize(ctx->stream));
    VQ_HIP(ctx, hipFree(d_ptr));
    return VQ_OK;
}

int32_t vq_host_alloc(vq_ctx *ctx, size_t bytes, void **h_ptr) {
    if (!ctx || !h_ptr) return VQ_ERR_INVALID_ARG;
    *h_ptr = nullptr;
    VQ_HIP(ctx, hipSetDevice(ctx->device));
    VQ_HIP(ctx, hipHostMalloc(h_ptr, bytes ? bytes : 1, hipHostMallocDefault));
    return VQ_OK;
}

int32_t vq_host_free(vq_ctx *ctx, void *h_ptr) {
    if (!ctx) return VQ_ERR_INVALID_ARG;
    if (!h_ptr) return VQ_OK;
    VQ_HIP(ctx, hipStreamSynchronize(ctx->stream));
    VQ_HIP(ctx, hipHostFree(h_ptr));
    return VQ_OK;
}

int32_t vq_timer_start(vq_ctx *ctx) {
    if (!ctx) return VQ_ERR_INVALID_ARG;
    VQ_HIP(ctx, hipEventRecord(ctx->ev0, ctx->stream));
    return VQ_OK;
}

int32_t vq_timer_stop(vq_ctx *ctx, float *h_ms) {
    if (!ctx || !h_ms) return VQ_ERR_INVALID_ARG;
    VQ_HIP(ctx, hipEventRecord(ctx->ev1, ctx->stream));
    VQ_HIP(ctx, hipEventSynchronize(ctx->ev1));
    VQ_HIP(ctx, hipEventElapsedTime(h_ms, ctx->ev0, ctx->ev1));
    return VQ_OK;
}

int32_t vq_calibrate(vq_ctx *ctx, int32_t what, double *h_rate) {
    if (!ctx || !h_rate) return VQ_ERR_INVALID_ARG;
    VQ_HIP(ctx, hipSetDevice(ctx->device));
    hipStream_t st = ctx->stream;
    float ms = 0.f;
    if (what == VQ_CALIB_HBM_COPY) {
        // 512 MB read + 512 MB written by the plain copy kernel, best of five
        const int64_t count = 128LL * 1000 * 1000;
        VQ_TRY(ensure(ctx, ctx->tmp_a, sizeof(float) * count));
        VQ_TRY(ensure(ctx, ctx->tmp_b, sizeof(float) * count));
        VQ_HIP(ctx, hipMemsetAsync(ctx->tmp_a.p, 0, sizeof(float) * count, st));
        float best = 1e30f;
        for (int rep = 0; rep < 6; ++rep) {
            VQ_HIP(ctx, hipEventRecord(ctx->ev0, st));
            VQ_TRY(vq_copy_f32(ctx, (float *)ctx->tmp_b.p, (const float *)ctx->tmp_a.p, count));
            VQ_HIP(ctx, hipEventRecord(ctx->ev1, st));
            VQ_HIP(ctx, hipEventSynchronize(ctx->ev1));
            VQ_HIP(ctx, hipEventElapsedTime(&ms, ctx->ev0, ctx->ev1));
            if (rep > 0 && ms < best) best = ms;
        }
        *h_rate = 2.0 * sizeof(float) * (double)count / (best * 1e-3) / 1e9;  // GB/s, read + write
        return VQ_OK;
    }
    if (what < VQ_CALIB_VALU_FMA || what > VQ_CALIB_VALU_ADD)
        return fail(ctx, VQ_ERR_INVALID_ARG, "Invalid parameter: calibration kind %d", what);
    hipDeviceProp_t prop;
    VQ_HIP(ctx, hipGetDeviceProperties(&prop, ctx->device));
    const int iters = 2048;
    const unsigned blocks = (unsigned)prop.multiProcessorCount * 8u;  // 8 waves on every SIMD
    VQ_TRY(ensure(ctx, ctx->tmp_a, 256));
    float best = 1e30f;
    for (int rep = 0; rep < 4; ++rep) {
        VQ_HIP(ctx, hipEventRecord(ctx->ev0, st));
        uint32_t *sink = (uint32_t *)ctx->tmp_a.p;
        switch (what) {
        case VQ_CALIB_VALU_FMA: hipLaunchKernelGGL(vq::k_calib_valu<0>, dim3(blocks), dim3(256), 0, st, iters, 1u, sink); break;
        case VQ_CALIB_VALU_MIN3: hipLaunchKernelGGL(vq::k_calib_valu<1>, dim3(blocks), dim3(256), 0, st, iters, 1u, sink); break;
        case VQ_CALIB_VALU_MED3: hipLaunchKernelGGL(vq::k_calib_valu<2>, dim3(blocks), dim3(256), 0, st, iters, 1u, sink); break;
        case VQ_CALIB_VALU_AND_OR: hipLaunchKernelGGL(vq::k_calib_valu<3>, dim3(blocks), dim3(256), 0, st, iters, 1u, sink); break;
        default: hipLaunchKernelGGL(vq::k_calib_valu<4>, dim3(blocks), dim3(256), 0, st, iters, 1u, sink); break;
        }
        VQ_HIP(ctx, hipGetLastError());
        VQ_HIP(ctx, hipEventRecord(ctx->ev1, st));
        VQ_HIP(ctx, hipEventSynchronize(ctx->ev1));
        VQ_HIP(ctx, hipEventElapsedTime(&ms, ctx->ev0, ctx->ev1));
        if (rep > 0 && ms < best) best = ms;
    }
    // wave64 instructions per second over the whole GPU
    const double instr = (double)blocks * 4.0 * iters * vq::kCalibChains * vq::kCalibUnroll;
    *h_rate = instr / (best * 1e-3);
    return VQ_OK;
}

int32_t vq_calibrate_overlap(vq_ctx *ctx, int32_t mode, double *h_ms, uint32_t *h_waves) {
    if (!ctx || !h_ms || mode < 0 || mode > 2)
        return fail(ctx, VQ_ERR_INVALID_ARG, "Invalid parameter: overlap calibration mode %d", mode);
    VQ_HIP(ctx, hipSetDevice(ctx->device));
    hipStream_t st = ctx->stream;
    hipDeviceProp_t prop;
    VQ_HIP(ctx, hipGetDeviceProperties(&prop, ctx->device));
    const unsigned waves_per_cu = 32u;  // 8 on every SIMD
    VQ_TRY(ensure(ctx, ctx->tmp_a, 256));
    uint32_t *sink = (uint32_t *)ctx->tmp_a.p, *where = sink + 8;
    const int n_mfma = 4096;
    const int vpm = mode == 0 ? 8 : mode == 1 ? 7 : 3;  // vector instructions per matrix instruction
    const int n_valu = n_mfma * vpm;
    for (int which = 0; which < 3; ++which) {
        const int nm = which == 1 ? 0 : n_mfma, nv = which == 0 ? 0 : n_valu;
        float best = 1e30f, ms = 0.f;
        for (int rep = 0; rep < 4; ++rep) {
            VQ_HIP(ctx, hipMemsetAsync(where, 0, 8 * sizeof(uint32_t), st));
            VQ_HIP(ctx, hipEventRecord(ctx->ev0, st));
            if (mode == 0)
                hipLaunchKernelGGL((vq::k_calib_overlap<0, 8>), dim3((unsigned)prop.multiProcessorCount * waves_per_cu / 8u),
                                   dim3(512), 0, st, nm, nv, 1u, sink, where);
            else if (mode == 1)
                hipLaunchKernelGGL((vq::k_calib_overlap<1, 7>), dim3((unsigned)prop.multiProcessorCount * waves_per_cu / 4u),
                                   dim3(256), 0, st, nm, nv, 1u, sink, where);
            else
                hipLaunchKernelGGL((vq::k_calib_overlap<1, 3>), dim3((unsigned)prop.multiProcessorCount * waves_per_cu / 4u),
                                   dim3(256), 0, st, nm, nv, 1u, sink, where);
            VQ_HIP(ctx, hipGetLastError());
            VQ_HIP(ctx, hipEventRecord(ctx->ev1, st));
            VQ_HIP(ctx, hipEventSynchronize(ctx->ev1));
            VQ_HIP(ctx, hipEventElapsedTime(&ms, ctx->ev0, ctx->ev1));
            if (rep > 0 && ms < best) best = ms;
        }
        h_ms[which] = best;
    }
    if (h_waves) {
        if (mode == 0) {
            VQ_HIP(ctx, hipMemcpyAsync(h_waves, where, 8 * sizeof(uint32_t), hipMemcpyDeviceToHost, st));
            VQ_HIP(ctx, hipStreamSynchronize(st));
        } else {
            for (int i = 0; i < 8; ++i) h_waves[i] = 0u;
        }
    }
    return VQ_OK;
}

int32_t vq_ctx_set_tsvq_variance_path(vq_ctx *ctx, int32_t path) {
    if (!ctx || (path != 0 && path != 1)) return VQ_ERR_INVALID_ARG;
    ctx->tsvq_var_path = path;
    return VQ_OK;
}

int32_t vq_ctx_set_assign_path(vq_ctx *ctx, int32_t path) {
    if (!ctx || (path != 0 && path != 1)) return VQ_ERR_INVALID_ARG;
    ctx->assign_path = path;
    return VQ_OK;
}

int32_t vq_ctx_set_few_path(vq_ctx *ctx, int32_t path) {
    if (!ctx || (path != 0 && path != 1)) return VQ_ERR_INVALID_ARG;
    ctx->few_path = path;
    return VQ_OK;
}

int32_t vq_ctx_last_recheck_count(vq_ctx *ctx, uint32_t *h_count) {
    if (!ctx || !h_count) return VQ_ERR_INVALID_ARG;
    uint32_t all = 0, two = 0;
    const int32_t rc = vq_ctx_last_recheck_split(ctx, &all, &two);
    *h_count = all + two;
    return rc;
}

int32_t vq_ctx_last_recheck_split(vq_ctx *ctx, uint32_t *h_count, uint32_t *h_two) {
    if (!ctx || !h_count || !h_two) return VQ_ERR_INVALID_ARG;
    *h_count = 0;
    *h_two = 0;
    if (ctx->recheck_src == 1 || ctx->recheck_src == 3) {
        uint32_t h[vq::kStatSlots * vq::kStatStride];
        const void *src = ctx->recheck_src == 1
                              ? (const void *)((uint32_t *)ctx->mfma_stat.p + ctx->mfma_stat_cur * vq::kStatSlots * vq::kStatStride)
                              : ctx->static_scratch + kNoAllocStatOff;
        VQ_HIP(ctx, hipMemcpyAsync(h, src, sizeof(h), hipMemcpyDeviceToHost, ctx->stream));
        VQ_HIP(ctx, hipStreamSynchronize(ctx->stream));
        for (int i = 0; i < vq::kStatSlots; ++i) *h_count += h[i * vq::kStatStride];
    } else if (ctx->recheck_src == 2) {
        uint32_t h[2];  // all-centroid checks, two-candidate checks
        VQ_HIP(ctx, hipMemcpyAsync(h, ctx->mfma_list.p, sizeof(h), hipMemcpyDeviceToHost, ctx->stream));
        VQ_HIP(ctx, hipStreamSynchronize(ctx->stream));
        *h_count = h[0];
        *h_two = h[1];
    }
    return VQ_OK;
}

int32_t vq_prof_enable(vq_ctx *ctx, int32_t on) {
    if (!ctx) return VQ_ERR_INVALID_ARG;
    VQ_HIP(ctx, hipStreamSynchronize(ctx->stream));
    prof_collect(ctx);
    ctx->prof_on = on != 0;
    for (int i = 0; i < VQ_PROF_CLASSES; ++i) {
        ctx->prof_ms[i] = 0;
        ctx->prof_launches[i] = 0;
    }
    return VQ_OK;
}

int32_t vq_prof_read(vq_ctx *ctx, int32_t cls, double *h_total_ms, int64_t *h_spans) {
    if (!ctx || cls < 0 || cls >= VQ_PROF_CLASSES || !h_total_ms || !h_spans)
        return VQ_ERR_INVALID_ARG;
    VQ_HIP(ctx, hipStreamSynchronize(ctx->stream));
    prof_collect(ctx);
    *h_total_ms = ctx->prof_ms[cls];
    *h_spans = ctx->prof_launches[cls];
    return VQ_OK;
}

int32_t vq_copy_f32(vq_ctx *ctx, float *d_dst, const float *d_src, int64_t count) {
    if (!ctx || count < 0 || (count && (!d_dst || !d_src))) return VQ_ERR_INVALID_ARG;
    if ((reinterpret_cast<uintptr_t>(d_dst) | reinterpret_cast<uintptr_t>(d_src)) & 15)
        return fail(ctx, VQ_ERR_INVALID_ARG, "Invalid parameter: buffers must be 16-byte aligned");
    if (count == 0) return VQ_OK;
    VQ_HIP(ctx, hipSetDevice(ctx->device));
    int64_t n4 = count / 4;
    int tail = (int)(count % 4);
    unsigned blocks = (unsigned)std::min<int64_t>(std::max<int64_t>((n4 + 255) / 256, 1), 256 * 32);
    hipLaunchKernelGGL(k_copy_f32, dim3(blocks), dim3(256), 0, ctx->stream, (const float4 *)d_src,
                       (float4 *)d_dst, n4, d_src + n4 * 4, d_dst + n4 * 4, tail);
    VQ_HIP(ctx, hipGetLastError());
    return VQ_OK;
}

}  // extern "C"

template <typename Last>
static int32_t lbg_fit_run(vq_ctx *ctx, const float *d_x, int64_t n, int64_t ld, int32_t m, int32_t sd, int32_t k,
                           int32_t max_iters, const uint32_t *h_init_idx, const uint32_t *h_reseed_stream,
                           int32_t n_reseed, float *d_codebooks, int32_t *h_iters_run, int32_t *h_reseeds_used,
                           const float *pend_cb, const uint8_t *pend_codes, bool residual, const Last &last);

// pend_cb / pend_codes: a residual update x[i] -= pend_cb[pend_codes[i]] that the fit applies to the
// rows in place as its first assignment pass reads them (the caller has checked that this shape's
// first pass is the kernel that can: lbg_pending_fusable).  residual: the rows are (or become so) what a stage left.
static int32_t lbg_fit_impl(vq_ctx *ctx, const float *d_x, int64_t n, int64_t ld, int32_t m, int32_t sd,
                            int32_t k, int32_t max_iters, const uint32_t *h_init_idx,
                            const uint32_t *h_reseed_stream, int32_t n_reseed, float *d_codebooks,
                            int32_t *h_iters_run, int32_t *h_reseeds_used, const float *pend_cb,
                            const uint8_t *pend_codes, bool residual) {
    if (!ctx) return VQ_ERR_INVALID_ARG;
    if (k == 0) return fail(ctx, VQ_ERR_INVALID_ARG, "Invalid parameter: k must be greater than 0");
    VQ_TRY(check_common(ctx, d_x, n, ld, m, sd, k, 65536));
    if (n < k)
        return fail(ctx, VQ_ERR_INVALID_ARG, "Invalid parameter: Not enough data points for k clusters");
    if (m > 65535) return fail(ctx, VQ_ERR_UNSUPPORTED, "m must be at most 65535");
    if (!h_init_idx || !d_codebooks || max_iters < 0 || n_reseed < 0 || (n_reseed && !h_reseed_stream))
        return fail(ctx, VQ_ERR_INVALID_ARG, "Invalid parameter: null pointer or negative size");
    for (int64_t i = 0; i < (int64_t)m * k; ++i)
        if (h_init_idx[i] >= (uint64_t)n)
            return fail(ctx, VQ_ERR_INVALID_ARG, "Invalid parameter: init index %u out of range", h_init_idx[i]);
    for (int64_t i = 0; i < (int64_t)m * n_reseed; ++i)
        if (h_reseed_stream[i] >= (uint64_t)n)
            return fail(ctx, VQ_ERR_INVALID_ARG, "Invalid parameter: reseed index %u out of range", h_reseed_stream[i]);
    VQ_HIP(ctx, hipSetDevice(ctx->device));
    if (k > vq::kMaxK) {
        // rows that every pass would pad, once for the fit, as below (200,131 x 36 blocks of 3, k = 280: 62 of 920 us per
        // iteration; 5,851 x 23 of 9, k = 1953: 97 of 400)
        const int w = max_iters > 0 ? encode_pad_width(ctx, VQ_SQEUCLIDEAN, d_x, n, ld, m, sd, vq::kMaxK, d_codebooks) : 0;
        if (w) {
            int32_t rc = ensure(ctx, ctx->pad_rows, sizeof(float) * ((size_t)n * m + (size_t)m * k) * w);
            if (rc == VQ_OK) {
                float *px = (float *)ctx->pad_rows.p, *pcb = px + (size_t)n * m * w;
                launch_pad(ctx, d_x, n, ld, m, sd, w, px);
                rc = vqh::lbg_fit_big(ctx, px, n, (int64_t)m * w, m, w, k, max_iters, h_init_idx, h_reseed_stream, n_reseed, pcb,
                                      h_iters_run, h_reseeds_used, [&] { unpad_rows(ctx, pcb, (int64_t)m * k, sd, w, d_codebooks); });
            }
            if (rc == VQ_ERR_OOM || ctx->pad_rows.cap > kPadKeep) {
                const int32_t gone = release(ctx, ctx->pad_rows);
                if (rc == VQ_OK) rc = gone;
            }
            if (rc != VQ_ERR_OOM) return rc;
        }
        return vqh::lbg_fit_big(ctx, d_x, n, ld, m, sd, k, max_iters, h_init_idx, h_reseed_stream, n_reseed,
                                d_codebooks, h_iters_run, h_reseeds_used);
    }
    vq::AssignArgs shape;
    shape.x = d_x;
    shape.n = n;
    shape.ld = ld;
    shape.m = m;
    shape.k = k;
    shape.cb = d_codebooks;
    const int sdp = max_iters > 0 ? pad_width(ctx, VQ_SQEUCLIDEAN, shape, sd, true, residual) : 0;
    if (sdp && (int64_t)k * cdiv(n, vq::kPartRows) * sdp <= (1LL << 31)) {
        // the rows padded once for all passes of the fit (where the second copy of the rows and the fit's
        // workspace do not fit together, it trains on the rows as they are: the same results)
        int32_t rc = ensure(ctx, ctx->pad_x, sizeof(float) * (size_t)n * m * sdp);
        if (rc == VQ_OK) rc = ensure(ctx, ctx->pad_cb, sizeof(float) * (size_t)m * k * sdp);
        if (rc == VQ_OK) {
            float *px = (float *)ctx->pad_x.p, *pcb = (float *)ctx->pad_cb.p;
            launch_pad(ctx, d_x, n, ld, m, sd, sdp, px);
            rc = lbg_fit_run(ctx, px, n, (int64_t)m * sdp, m, sdp, k, max_iters, h_init_idx, h_reseed_stream, n_reseed,
                             pcb, h_iters_run, h_reseeds_used, nullptr, nullptr, residual, [&] {
                                 unpad_rows(ctx, pcb, (int64_t)m * k, sd, sdp, d_codebooks);
                             });
        }
        // a large copy is not held for later calls (taking 2.3 GB again costs a fit of 1,500,000 x 96 in
        // blocks of 2 0.8 ms of 18)
        if (rc == VQ_ERR_OOM || ctx->pad_x.cap > kPadKeep) {
            const int32_t gone = release(ctx, ctx->pad_x);
            if (rc == VQ_OK) rc = gone;
        }
        if (rc != VQ_ERR_OOM) return rc;
    }
    return lbg_fit_run(ctx, d_x, n, ld, m, sd, k, max_iters, h_init_idx, h_reseed_stream, n_reseed, d_codebooks,
                       h_iters_run, h_reseeds_used, pend_cb, pend_codes, residual, [] {});
}

// Clusters per workgroup of k_lbg_update_small: the fewest with which the workgroups (106 KB of LDS each) are one
// round of the 256 compute units, as far as one thread per (cluster, component) and four bits per list entry
// allow.  (m = 10, k = 200, 60,007 rows: 7 clusters are 290 workgroups and 64 us, 8 are 250 and 42 us.)
static int lbg_small_clusters(int m, int sd, int k) {
    const int most = std::max(1, std::min(vq::kSmallClusters, (sd <= vq::kSmallThreads ? vq::kSmallThreads : 4096) / sd));
    int c = 1;
    while (c < most && (int64_t)m * ((k + c - 1) / c) > 256) ++c;
    return c;
}

// Components of a workgroup of k_lbg_update_small: blocks above 32 floats are taken by tiles of 16 or 32 where those are a
// round of the GPU; the last tile begins at the block's end less its width.
static int lbg_small_width(int m, int sd, int k) {
    if (sd <= 32) return sd;
    for (int w : {16, 32})
        if ((int64_t)m * (int64_t)cdiv(sd, w) * (int64_t)cdiv(k, vq::kSmallClusters) <= 256) return w;
    return sd;
}

// Whether the update of a fit runs as k_lbg_update_small.  Its time follows the members of a cluster
// (one chain of additions each) and the floats that a workgroup brings in, the other path's the number
// of its launches.  The two take the same time near 700 members where the chain decides (blocks of
// 8 floats, k = 116) and near 75,000 floats per workgroup in narrow blocks, 45,000-70,000 in wide ones, on
// uniform rows and on mixtures.  Ten iterations, m = 16, k = 256, blocks of 8: 2,000 rows 0.83 -> 0.22 ms,
// 10,000 1.07 -> 0.29 ms, 50,000 1.35 -> 0.74 ms; m = 1, k = 256, 20,000 x 128: 0.78 -> 0.45 ms.
// A block that is the whole row (m == 1).  What decides is the longest cluster: even rows keep the clusters even in every
// stage, the residuals of clustered rows gather in a few of them, and every workgroup lists all rows.  So the lines lie lower where
// the rows are what a stage left, where both kinds of rows lose as much on one side as on the other.  A fit of five iterations, k = 256, other
// path -> this one: uniform rows, first stage 52,428 x 24 307 -> 227 us, 78,643 x 32 337 -> 273, 52,428 x 64 355 -> 298, 78,643 389 -> 410, 32,768 x
// 128 405 -> 331, 65,536 452 -> 441; a mixture of 1024 Gaussians, first stage 104,857 x 24 365 -> 372, 52,428 x 64 374 -> 323, 78,643 402 -> 529.
// Residuals: uniform 52,428 x 24 305 -> 234, 78,643 328 -> 314, 52,428 x 64 360 -> 304, 78,643 392 -> 412, 28,086 x 224 446 -> 417; mixture 52,428 x
// 24 322 -> 360, 78,643 357 -> 477, 32,768 x 64 337 -> 360, 52,428 365 -> 460, 28,086 x 224 451 -> 518, 131,072 x 64 441 -> 1377.  k = 64, residuals of a
// mixture: 32,768 x 64 1.02 times the other path's time, 40,960 1.19, 9,361 x 224 1.00; uniform 0.75, 0.86, 0.77.  Above 160 floats the residuals'
// line is a number of floats.
// Several wide blocks: their rows spread over the clusters too.  Fit of five iterations and encode: two blocks of 48, k = 256 33,000 rows
// 400 -> 345, 40,000 393 -> 358, 48,000 404 -> 385, 65,000 468 -> 508, k = 128 36,000 364 -> 356, 44,000 371 -> 395; three of 36, k = 180 36,000 424 -> 396,
// 44,000 448 -> 434, k = 100 33,000 429 -> 388, 40,000 423 -> 439; four of 64, k = 256 36,000 465 -> 439, 44,000 495 -> 502, k = 180 33,000 466 -> 447,
// 36,000 467 -> 499; two of 96, k = 256 36,000 435 -> 404, 44,000 457 -> 520; two of 128, k = 256 33,000 498 -> 513, 40,000 492 -> 523.
static bool lbg_small(int64_t n, int m, int sd, int k, bool residual) {
    if (sd % 4 != 0 || sd > 4096 || n > 131072) return false;
    if (sd > vq::kSmallThreads) return n <= 128 * (int64_t)k;
    if (n > 640 * (int64_t)k || n * lbg_small_clusters(m, sd, k) * sd > (sd <= 32 ? 57344 : 40960) * (int64_t)k) return false;
    if (m > 1) return sd <= 32 || n <= std::max(32768, sd > 96 ? 0 : sd <= 48 ? 27000 + 90 * k : 24000 + 62 * k);
    if (sd < 16) return true;
    if (residual)
        return sd > 160 ? n * sd <= 3'600'000 : n <= (sd == 16 ? 104'000 : sd <= 32 ? 36000 + 70 * k : sd <= 64 ? 28000 + 90 * k : 25000 + 50 * k);
    return sd == 16 || n <= (sd <= 32 ? 30000 + 280 * k : sd <= 64 ? 35000 + 95 * k : 30000 + 70 * k);
}

// The LBG loop of a small fit, two launches per iteration: the assignment and k_lbg_update_small.  The
// index streams stay in page-locked host memory: the initial rows are read once, re-seed rows rarely.
template <typename Last>
static int32_t lbg_fit_small(vq_ctx *ctx, const float *d_x, int64_t n, int64_t ld, int32_t m, int32_t sd, int32_t k,
                             int32_t max_iters, const uint32_t *h_init_idx, const uint32_t *h_reseed_stream,
                             int32_t n_reseed, float *d_codebooks, int32_t *h_iters_run, int32_t *h_reseeds_used,
                             const float *pend_cb, const uint8_t *pend_codes, const Last &last) {
    hipStream_t st = ctx->stream;
    const size_t n_flags = (2 * (size_t)max_iters + 1) * m + 1, n_idx = (size_t)m * k, n_res = (size_t)m * n_reseed;
    // wide blocks: clusters above 1024 members by k_lbg_large (one more launch per iteration; up to two
    // parts of rows there is nothing to gain)
    const bool staged = sd <= vq::kSmallThreads;
    const int nparts = (int)cdiv(n, vq::kPartRows);
    const bool defer = staged && sd > 32 && nparts > 2;
    const int width = staged ? lbg_small_width(m, sd, k) : sd, tiles = (int)cdiv(sd, width);
    const int most_large = defer ? (int)(m * (n / (vq::kSeqMax + 1))) : 0;
    VQ_TRY(ensure(ctx, ctx->flags, sizeof(int) * (n_flags + max_iters + (size_t)most_large * tiles)));
    VQ_TRY(ensure(ctx, ctx->codes, (size_t)m * n + 4));
    if (defer) {
        VQ_TRY(ensure(ctx, ctx->leaf_desc, sizeof(uint2) * (size_t)most_large));
        VQ_TRY(ensure(ctx, ctx->leaf_sum, sizeof(float) * (size_t)most_large * nparts * sd));
    }
    VQ_TRY(ensure_pinned(ctx, ctx->lbg_pin, ctx->lbg_pin_cap, sizeof(uint32_t) * (n_idx + n_res + n_flags)));
    uint32_t *idx = (uint32_t *)ctx->lbg_pin, *reseed = idx + n_idx;
    int *report = (int *)(reseed + n_res);
    memcpy(idx, h_init_idx, sizeof(uint32_t) * n_idx);
    if (n_res) memcpy(reseed, h_reseed_stream, sizeof(uint32_t) * n_res);
    vq::LbgSmall S;
    S.changed = (int *)ctx->flags.p;
    S.empties = S.changed + (size_t)(max_iters + 1) * m;
    S.err = S.empties + (size_t)max_iters * m;
    S.codes = (uint8_t *)ctx->codes.p;
    S.n_large = S.err + 1;
    S.arrived = S.n_large + max_iters;
    S.large = (uint2 *)ctx->leaf_desc.p;
    S.large_sum = (float *)ctx->leaf_sum.p;
    const int64_t init_items = std::max<int64_t>((int64_t)m * k * sd, (int64_t)m * n / 4);
    hipLaunchKernelGGL(vq::k_lbg_small_init, dim3(std::min<unsigned>(cdiv(init_items, 256), 1024u)), dim3(256), 0, st, S,
                       d_x, n, ld, m, k, sd, max_iters, most_large * tiles, (const uint32_t *)idx, d_codebooks, pend_cb, pend_codes);
    vq::AssignArgs a;
    a.x = d_x;
    a.n = n;
    a.ld = ld;
    a.m = m;
    a.k = k;
    a.cb = d_codebooks;
    a.cnorm = nullptr;
    a.codes = S.codes;
    a.done = nullptr;
    const int C = lbg_small_clusters(m * tiles, width, k);
    const int groups = (int)cdiv(k, C);
    if (staged && !ctx->lbg_small_lds_set) {
        const void *kerns[] = {reinterpret_cast<const void *>(vq::k_lbg_update_small<true>),
                               reinterpret_cast<const void *>(vq::k_lbg_update_small<true, false, 8>),
                               reinterpret_cast<const void *>(vq::k_lbg_update_small<true, false, 16>),
                               reinterpret_cast<const void *>(vq::k_lbg_update_small<true, false, 32>),
                               reinterpret_cast<const void *>(vq::k_lbg_update_small<true, true>),
                               reinterpret_cast<const void *>(vq::k_lbg_update_small<true, false, 16, true>),
                               reinterpret_cast<const void *>(vq::k_lbg_update_small<true, false, 32, true>),
                               reinterpret_cast<const void *>(vq::k_lbg_update_small<true, true, 16, true>),
                               reinterpret_cast<const void *>(vq::k_lbg_update_small<true, true, 32, true>),
                               reinterpret_cast<const void *>(vq::k_lbg_large<0>),
                               reinterpret_cast<const void *>(vq::k_lbg_large<16>),
                               reinterpret_cast<const void *>(vq::k_lbg_large<32>)};
        for (const void *kern : kerns)
            VQ_HIP(ctx, hipFuncSetAttribute(kern, hipFuncAttributeMaxDynamicSharedMemorySize,
                                            (int)(sizeof(float) * vq::kSmallStage)));
        ctx->lbg_small_lds_set = true;
    }
    for (int it = 0; it < max_iters; ++it) {
        a.pend_cb = it == 0 ? pend_cb : nullptr;  // the first pass leaves the rows updated
        a.pend_codes = it == 0 ? pend_codes : nullptr;
        a.before = S.changed + (size_t)it * m;
        a.changed = S.changed + (size_t)(it + 1) * m;
        {
            ProfSpan sp(ctx, VQ_PROF_LBG_ASSIGN);
            VQ_TRY(launch_assign<true>(ctx, VQ_SQEUCLIDEAN, a, sd));
        }
        ProfSpan sp(ctx, VQ_PROF_LBG_UPDATE);
        const unsigned wgs = (unsigned)groups * m * tiles;
        const size_t lds = sizeof(float) * (staged ? vq::kSmallStage : 3 * (size_t)C * sd);
        const auto tiled = width == 16 ? (defer ? vq::k_lbg_update_small<true, true, 16, true> : vq::k_lbg_update_small<true, false, 16, true>)
                                       : (defer ? vq::k_lbg_update_small<true, true, 32, true> : vq::k_lbg_update_small<true, false, 32, true>);
        const auto kern = !staged    ? vq::k_lbg_update_small<false>
                          : tiles > 1 ? tiled
                          : sd == 8   ? vq::k_lbg_update_small<true, false, 8>
                          : sd == 16  ? vq::k_lbg_update_small<true, false, 16>
                          : sd == 32  ? vq::k_lbg_update_small<true, false, 32>
                          : defer     ? vq::k_lbg_update_small<true, true>
                                      : vq::k_lbg_update_small<true>;
        hipLaunchKernelGGL(kern, dim3(wgs), dim3(vq::kSmallThreads), lds, st, S, it, m, d_x, n, ld, sd, k, C, groups,
                           (const uint32_t *)reseed, n_reseed, d_codebooks, tiles);
        const int whole = std::min(most_large, 16);
        if (defer)
            hipLaunchKernelGGL(width == 16 ? vq::k_lbg_large<16> : width == 32 ? vq::k_lbg_large<32> : vq::k_lbg_large<0>, dim3(nparts, whole + (tiles > 1 ? vq::kLargeTurns * tiles : 0)),
                               dim3(vq::kSmallThreads), lds, st, S, it, d_x, n, ld, sd, k, whole, d_codebooks);
    }
    last();
    hipLaunchKernelGGL(vq::k_lbg_small_report, dim3(1), dim3(256), 0, st, (const int *)S.changed, (int)n_flags, report);
    VQ_HIP(ctx, hipGetLastError());
    VQ_HIP(ctx, hipStreamSynchronize(st));
    prof_collect(ctx);
    const int *changed = report, *empties = report + (size_t)(max_iters + 1) * m;
    for (int s = 0; s < m; ++s) {
        int iters = 0, used = 0;
        for (int it = 0; it < max_iters && changed[(size_t)it * m + s]; ++it) {
            ++iters;
            used += empties[(size_t)it * m + s];
        }
        if (h_iters_run) h_iters_run[s] = iters;
        if (h_reseeds_used) h_reseeds_used[s] = used;
    }
    if (report[n_flags - 1])
        return fail(ctx, VQ_ERR_RESEED_EXHAUSTED, "re-seed stream exhausted: pass n_reseed = k*max_iters");
    return VQ_OK;
}

// The LBG loop for up to 256 centroids, on validated arguments.  last: enqueues what follows the
// last update, before the loop's results are read back.
template <typename Last>
static int32_t lbg_fit_run(vq_ctx *ctx, const float *d_x, int64_t n, int64_t ld, int32_t m, int32_t sd, int32_t k,
                           int32_t max_iters, const uint32_t *h_init_idx, const uint32_t *h_reseed_stream,
                           int32_t n_reseed, float *d_codebooks, int32_t *h_iters_run, int32_t *h_reseeds_used,
                           const float *pend_cb, const uint8_t *pend_codes, bool residual, const Last &last) {
    if (lbg_small(n, m, sd, k, residual))
        return lbg_fit_small(ctx, d_x, n, ld, m, sd, k, max_iters, h_init_idx, h_reseed_stream, n_reseed, d_codebooks,
                             h_iters_run, h_reseeds_used, pend_cb, pend_codes, last);
    hipStream_t st = ctx->stream;

    const int nparts = (int)((n + vq::kPartRows - 1) / vq::kPartRows);
    const int nseg = (nparts + vq::kScanSeg - 1) / vq::kScanSeg;
    // streaming sums of the large clusters: 32-byte sub-vectors, 4 to a workgroup, aligned rows
    const bool stream = sd == 8 && stream_pays(n, m, k) && ld % 4 == 0 && ld <= (1 << 20) &&
                        (reinterpret_cast<uintptr_t>(d_x) & 15) == 0;  // (32-bit lane offsets inside a chunk)
    const int64_t leaf_cap64 = stream ? (int64_t)k : (int64_t)k * nparts;
    if (leaf_cap64 * sd > (1LL << 31)) return fail(ctx, VQ_ERR_UNSUPPORTED, "n * k * sub_dim too large");
    const int leaf_cap = (int)leaf_cap64;
    VQ_TRY(ensure(ctx, ctx->flags, sizeof(int) * (8 * (size_t)m + 1)));
    VQ_TRY(ensure(ctx, ctx->tables, sizeof(uint32_t) * 4 * (size_t)m * vq::kMaxK));
    VQ_TRY(ensure(ctx, ctx->hist, sizeof(uint32_t) * (size_t)m * nparts * vq::kMaxK));
    VQ_TRY(ensure(ctx, ctx->seg, sizeof(uint32_t) * (size_t)m * nseg * vq::kMaxK));
    VQ_TRY(ensure(ctx, ctx->perm, sizeof(uint32_t) * (size_t)m * n));
    // per-part sums of the streaming kernel, then one folded sum per cluster
    if (stream) VQ_TRY(ensure(ctx, ctx->part_sum, sizeof(float) * (size_t)m * (nparts + 1) * vq::kMaxK * 8));
    // Blocks of 64 to 512 floats: leaves handed out long ones first, then part by part (k_lbg_leafsum_wide)
    // where the rows are well beyond the memory-side cache (256 MB): the order costs 5 us per iteration in the scan, and rows
    // that lie in the cache may be read in any order.  An iteration of a residual fit, k = 256, without -> with:
    // 150,000 x 256 172 -> 179 us, 300,000 240 -> 241, 500,000 351 -> 343, 1,000,000 620 -> 589; x 128: 300,000 164 -> 169, 600,000
    // 258 -> 252 (k = 121 2 % slower), 1,000,000 384 -> 360; x 512: 250,000 384 -> 390, 500,000 646 -> 633; 3,000,000 x 64 589 -> 565.
    const bool wide_leaves = !stream && sd >= 64 && sd <= 512 && n >= 300'000 && n * m * sd >= 100'000'000;
    // Else a workgroup per leaf and 32 components (k_lbg_leafsum_tile), of one wave where the leaves are parts of under 64
    // members (500,000 x 8 blocks of 16, k = 160: 284 us per iteration, with two waves 341, a lane per component 309; 50,019 x 28 of
    // 10, k = 78: two waves 141, one 142, a wave of 4-byte loads per leaf 223; 100,000 x 32, k = 128: 75, 83, a lane 155),
    // but a lane per component where leaves of under 20 members fill the GPU that way (600,000 x 12 of 16, k = 256: 525
    // against 583; 1M x 32, k = 256, on the other side: 221 and 198).
    const bool parted = n > (int64_t)vq::kSeqMax * k;  // an average cluster is summed part by part
    const bool lane_leaves = parted && vq::kPartRows < 20 * k && leaf_cap64 * sd * m >= (1 << 22);
    const size_t long_cap = (size_t)(n / vq::kLong + 1), leaf_slots = (size_t)m * leaf_cap;
    if (wide_leaves)  // the leaves in order, the two lists of long ones, the places, the counters
        VQ_TRY(ensure(ctx, ctx->leaf_desc, sizeof(uint4) * (leaf_slots + 2 * (size_t)m * long_cap) +
                                               sizeof(uint32_t) * (size_t)m * (vq::kMaxK + 2)));
    else
        VQ_TRY(ensure(ctx, ctx->leaf_desc, sizeof(uint2) * leaf_slots));
    VQ_TRY(ensure(ctx, ctx->leaf_sum, sizeof(float) * (size_t)m * leaf_cap * sd));
    VQ_TRY(ensure(ctx, ctx->codes, (size_t)m * n));
    VQ_TRY(ensure(ctx, ctx->idx, sizeof(uint32_t) * (size_t)m * k));
    VQ_TRY(ensure(ctx, ctx->reseed, sizeof(uint32_t) * ((size_t)m * n_reseed + 1)));

    vq::LbgState S;
    int *f = (int *)ctx->flags.p;
    S.changed = f;
    S.done = f + m;
    S.iters = f + 2 * m;
    S.used = f + 3 * m;
    S.ubase = f + 4 * m;
    S.nleaves = f + 5 * m;
    S.nsmall = f + 6 * m;
    S.err = f + 7 * m;
    S.done_next = f + 7 * m + 1;
    uint32_t *tb = (uint32_t *)ctx->tables.p;
    const size_t mk = (size_t)m * vq::kMaxK;
    S.count = tb;
    S.start = tb + mk;
    S.leaf_start = tb + 2 * mk;
    S.empty_rank = tb + 3 * mk;
    S.hist = (uint32_t *)ctx->hist.p;
    S.seg = (uint32_t *)ctx->seg.p;
    S.perm = (uint32_t *)ctx->perm.p;
    S.leaf_desc = (uint2 *)ctx->leaf_desc.p;
    S.leaf_sum = (float *)ctx->leaf_sum.p;
    S.part_sum = stream ? (float *)ctx->part_sum.p : nullptr;
    S.codes = (uint8_t *)ctx->codes.p;
    S.nparts = nparts;
    S.nseg = nseg;
    S.leaf_cap = leaf_cap;
    S.stream = stream ? 1 : 0;
    if (wide_leaves) {
        S.order = (uint4 *)ctx->leaf_desc.p;
        S.longs = S.order + leaf_slots;
        S.place = (uint32_t *)(S.longs + 2 * (size_t)m * long_cap);
        S.nlong = (int *)(S.place + (size_t)m * vq::kMaxK);
        S.long_cap = (int)long_cap;
    }

    VQ_HIP(ctx, hipMemcpyAsync(ctx->idx.p, h_init_idx, sizeof(uint32_t) * (size_t)m * k,
                               hipMemcpyHostToDevice, st));
    if (n_reseed)
        VQ_HIP(ctx, hipMemcpyAsync(ctx->reseed.p, h_reseed_stream,
                                   sizeof(uint32_t) * (size_t)m * n_reseed, hipMemcpyHostToDevice, st));
    VQ_HIP(ctx, hipMemsetAsync(S.codes, 0, (size_t)m * n, st));  // assignments = vec![0; n], utils.rs:55
    hipLaunchKernelGGL(vq::k_lbg_init, dim3(cdiv(m, 64)), dim3(64), 0, st, S, m);
    if (pend_cb)
        hipLaunchKernelGGL(vq::k_gather_rows_pend, dim3(cdiv((int64_t)k * sd, 256)), dim3(256), 0, st, d_x, ld, k, sd,
                           (const uint32_t *)ctx->idx.p, d_codebooks, pend_cb, pend_codes);
    else
        hipLaunchKernelGGL(vq::k_gather_rows, dim3(cdiv((int64_t)m * k * sd, 256)), dim3(256), 0, st, d_x,
                           ld, m, k, sd, (const uint32_t *)ctx->idx.p, d_codebooks);
    VQ_HIP(ctx, hipGetLastError());

    vq::AssignArgs a;
    a.x = d_x;
    a.n = n;
    a.ld = ld;
    a.m = m;
    a.k = k;
    a.cb = d_codebooks;
    a.cnorm = nullptr;
    a.codes = S.codes;
    a.changed = S.changed;
    a.done = S.done;

    // With the streaming sums and the matrix-core assignment, one kernel ends the update: the new
    // centroids, the loop control and the tables of the next assignment pass.
    const bool fused_tail = stream && mfma_applicable<vq::M_SQ, true>(ctx, a, sd);
    MfmaTabPtrs tabs{};
    if (fused_tail) {
        VQ_TRY(mfma_tab_ptrs(ctx, m, k, tabs));
        S.done_next = nullptr;
    }
    // Timing classes of the loop: where the assignment kernel carries its own events (started,
    // done) the assignment span is the kernel's and an update span runs from one kernel's end to
    // the next one's start, so nothing is recorded between the kernels of an iteration.
    hipEvent_t prev_done = nullptr;
    for (int it = 0; it < max_iters; ++it) {
        hipEvent_t started = nullptr, done = nullptr;
        a.pend_cb = it == 0 ? pend_cb : nullptr;  // the first pass leaves the rows updated
        a.pend_codes = it == 0 ? pend_codes : nullptr;
        {
            ProfSpan sp(ctx, fused_tail ? -1 : VQ_PROF_LBG_ASSIGN);
            VQ_TRY(launch_assign<true>(ctx, VQ_SQEUCLIDEAN, a, sd, fused_tail && it > 0, &started, &done));
        }
        if (ctx->prof_on && started && done) {
            ctx->prof_open.push_back({VQ_PROF_LBG_ASSIGN, started, done, false, false});
            if (prev_done) ctx->prof_open.push_back({VQ_PROF_LBG_UPDATE, prev_done, started, false, false});
        }
        prev_done = done;
        ProfSpan sp(ctx, fused_tail ? -1 : VQ_PROF_LBG_UPDATE);
        int shift = 0;
        while ((1 << shift) < sd) ++shift;
        const bool leaf_wg = stream && sd >= 4 && sd <= 32 && (1 << shift) == sd && ld % 4 == 0 &&
                             (reinterpret_cast<uintptr_t>(d_x) & 15) == 0;
        // The gather path of the small clusters needs only the new codes: with the streaming sums
        // it runs on the second stream beside them (a chain of short, latency-bound kernels next to
        // one long pass over the rows), and the two meet again before the large clusters' fold.
        hipStream_t gs = stream ? ctx->side : st;
        if (stream) {
            if (!done) {  // the assignment kernel carried no event
                VQ_HIP(ctx, hipEventRecord(ctx->ev_fork, st));
                done = ctx->ev_fork;
            }
            VQ_HIP(ctx, hipStreamWaitEvent(gs, done, 0));
            hipLaunchKernelGGL(vq::k_lbg_stream8, dim3(nparts, cdiv(m, 4)), dim3(256), 0, st, S, d_x, n, ld, m);
        }
        if (stream)
            hipLaunchKernelGGL(vq::k_lbg_hist, dim3(nparts, m), dim3(64), 0, gs, S, n);
        else
            hipLaunchKernelGGL(vq::k_lbg_hist_wg, dim3(nparts, m), dim3(256), 0, gs, S, n);
        if (!stream && nseg <= vq::kScanMost && !wide_leaves) {
            hipLaunchKernelGGL(vq::k_lbg_scan, dim3(m), dim3(256 * nseg), 0, gs, S, k);
        } else {
            hipLaunchKernelGGL(vq::k_lbg_scan_seg, dim3(nseg, m), dim3(256), 0, gs, S);
            hipLaunchKernelGGL(vq::k_lbg_plan, dim3(m), dim3(256), 0, gs, S, k);
            hipLaunchKernelGGL(vq::k_lbg_scan_blocks, dim3(nseg, m), dim3(256), 0, gs, S);
        }
        if (stream)  // beside the streaming kernel: one wave per part (four waves per part take its resources: 40 us, and 15 us more for the streaming kernel)
            hipLaunchKernelGGL(vq::k_lbg_scatter, dim3(nparts, m), dim3(64), 0, gs, S, n);
        else  // every row is listed: sixteen waves per part (four: 3-5 us more of an iteration)
            hipLaunchKernelGGL(vq::k_lbg_scatter_wg, dim3(nparts, m), dim3(64 * vq::kScatterWaves), 0, gs, S, n);
        if (leaf_wg) {
            // leaves are the few clusters of up to 1024 members beside the streaming kernel
            hipLaunchKernelGGL(vq::k_lbg_leafsum_wg, dim3(leaf_cap, m), dim3(256), 0, gs, S, d_x, n, ld, sd,
                               shift);
        } else if (wide_leaves) {
            // a workgroup per place and per long leaf; a block above 256 floats in two halves
            const int z = sd > 256 ? 2 : 1, threads = (int)cdiv(cdiv(sd, z), 64) * 64;
            hipLaunchKernelGGL(vq::k_lbg_leafsum_wide, dim3((unsigned)(leaf_cap + long_cap), m, z), dim3(threads), 0, gs, S, d_x,
                               n, ld, sd);
        } else if (!lane_leaves) {
            const int tiles = (int)cdiv(sd, 32), width = tiles == 1 ? sd : (int)cdiv(cdiv(sd, tiles), 4) * 4;
            const int threads = parted && vq::kPartRows < 64 * k ? 64 : 128, vec = sd >= 4 ? 4 : 1, pieces = (int)cdiv(width, vec);
            const size_t lds = sizeof(float) * (size_t)width * (8 * (threads / pieces) + 4);
            const dim3 grid(leaf_cap, m, (unsigned)cdiv(sd, width));
            auto *kern = threads == 64 ? (vec == 4 ? vq::k_lbg_leafsum_tile<64, 4> : vq::k_lbg_leafsum_tile<64, 1>)
                                       : (vec == 4 ? vq::k_lbg_leafsum_tile<128, 4> : vq::k_lbg_leafsum_tile<128, 1>);
            hipLaunchKernelGGL(kern, grid, dim3(threads), lds, gs, S, d_x, n, ld, sd, width, pieces);
        } else {
            hipLaunchKernelGGL(vq::k_lbg_leafsum, dim3(cdiv((int64_t)leaf_cap * sd, 256), m), dim3(256), 0, gs,
                               S, d_x, n, ld, sd);
        }
        float *big_sum = stream ? S.part_sum + (size_t)m * nparts * vq::kMaxK * 8 : nullptr;
        if (fused_tail)  // needs the streaming kernel only: in flight while the gather path ends
            hipLaunchKernelGGL(vq::k_lbg_fold8, dim3(cdiv((int64_t)k * 8, 256), m), dim3(256), 0, st, S, k, big_sum);
        if (stream) {
            VQ_HIP(ctx, hipEventRecord(ctx->ev_join, gs));
            VQ_HIP(ctx, hipStreamWaitEvent(st, ctx->ev_join, 0));
            if (!fused_tail)
                hipLaunchKernelGGL(vq::k_lbg_combine8, dim3(cdiv((int64_t)k * 8, 256), m), dim3(256), 0, st, S, k,
                                   d_codebooks);
        }
        if (fused_tail) {
            hipLaunchKernelGGL(vq::k_lbg_finalize_prep8, dim3(m), dim3(256), 0, st, S, d_x, ld, k,
                               (const uint32_t *)ctx->reseed.p, n_reseed, d_codebooks, (const float *)big_sum,
                               tabs.nb, tabs.atab, tabs.aux, tabs.stat, tabs.stat_next);
        } else {
            hipLaunchKernelGGL(vq::k_lbg_finalize, dim3(cdiv((int64_t)k * sd, 256), m), dim3(256), 0, st, S,
                               d_x, ld, k, sd, (const uint32_t *)ctx->reseed.p, n_reseed, d_codebooks);
            std::swap(S.done, S.done_next);
            a.done = S.done;
        }
        VQ_HIP(ctx, hipGetLastError());
    }
    if (ctx->prof_on && fused_tail && prev_done) {  // the last update: up to an event recorded here
        hipEvent_t end = prof_event(ctx);
        VQ_HIP(ctx, hipEventRecord(end, st));
        ctx->prof_open.push_back({VQ_PROF_LBG_UPDATE, prev_done, end, false, true});
    }
    last();
    std::vector<int> host(7 * (size_t)m + 1);
    VQ_HIP(ctx, hipMemcpyAsync(host.data(), f, sizeof(int) * host.size(), hipMemcpyDeviceToHost, st));
    VQ_HIP(ctx, hipStreamSynchronize(st));
    prof_collect(ctx);
    if (h_iters_run) memcpy(h_iters_run, host.data() + 2 * m, sizeof(int) * m);
    if (h_reseeds_used) memcpy(h_reseeds_used, host.data() + 3 * m, sizeof(int) * m);
    if (host[7 * (size_t)m])
        return fail(ctx, VQ_ERR_RESEED_EXHAUSTED,
                    "re-seed stream exhausted: pass n_reseed = k*max_iters");
    return VQ_OK;
}

extern "C" {

int32_t vq_lbg_fit(vq_ctx *ctx, const float *d_x, int64_t n, int64_t ld, int32_t m, int32_t sd,
                   int32_t k, int32_t max_iters, const uint32_t *h_init_idx,
                   const uint32_t *h_reseed_stream, int32_t n_reseed, float *d_codebooks,
                   int32_t *h_iters_run, int32_t *h_reseeds_used) {
    return lbg_fit_impl(ctx, d_x, n, ld, m, sd, k, max_iters, h_init_idx, h_reseed_stream, n_reseed, d_codebooks,
                        h_iters_run, h_reseeds_used, nullptr, nullptr, false);
}

int32_t vq_lbg_fit_residual(vq_ctx *ctx, float *d_res, int64_t n, int64_t ld, int32_t dim, int32_t k,
                            int32_t max_iters, const uint32_t *h_init_idx, const uint32_t *h_reseed_stream,
                            int32_t n_reseed, float *d_codebook, const float *d_prev_codebook, int32_t k_prev,
                            const uint8_t *d_prev_codes, int32_t *h_iters_run, int32_t *h_reseeds_used) {
    if (!ctx) return VQ_ERR_INVALID_ARG;
    if (!d_prev_codebook || !d_prev_codes || k_prev <= 0 || k_prev > 256)
        return fail(ctx, VQ_ERR_INVALID_ARG, "Invalid parameter: the previous stage's codebook and codes");
    // The first assignment pass can apply the update as it reads the rows when it is the matrix-core
    // pass over one wide column block and there is a first pass; the arguments the fused path does
    // not check itself are checked by the two calls of the other path.
    vq::AssignArgs a;
    a.x = d_res;
    a.n = n;
    a.ld = ld;
    a.m = 1;
    a.k = k;
    a.cb = d_codebook;
    const bool fusable = d_res && d_codebook && n >= k && k >= 1 && k <= vq::kMaxK && dim >= 16 && ld >= dim &&
                         max_iters >= 1 && (reinterpret_cast<uintptr_t>(d_prev_codebook) & 15) == 0 &&
                         mfma_wide_applicable<vq::M_SQ, true>(ctx, a, dim) &&
                         !mfma_applicable<vq::M_SQ, true>(ctx, a, dim);
    if (!fusable) {
        VQ_TRY(vq_residual_sub(ctx, d_res, n, ld, dim, k_prev, d_prev_codebook, d_prev_codes));
        return lbg_fit_impl(ctx, d_res, n, ld, 1, dim, k, max_iters, h_init_idx, h_reseed_stream, n_reseed,
                            d_codebook, h_iters_run, h_reseeds_used, nullptr, nullptr, true);
    }
    return lbg_fit_impl(ctx, d_res, n, ld, 1, dim, k, max_iters, h_init_idx, h_reseed_stream, n_reseed, d_codebook,
                        h_iters_run, h_reseeds_used, d_prev_codebook, d_prev_codes, true);
}

int32_t vq_assign(vq_ctx *ctx, int32_t metric, const float *d_x, int64_t n, int64_t ld, int32_t m,
                  int32_t sd, int32_t k, const float *d_codebooks, uint8_t *d_codes) {
    return vqh::assign_codes(ctx, metric, d_x, n, ld, m, sd, k, d_codebooks, d_codes);
}

int32_t vq_assign_noalloc(vq_ctx *ctx, int32_t metric, const float *d_x, int64_t n, int64_t ld, int32_t m,
                          int32_t sd, int32_t k, const float *d_codebooks, uint8_t *d_codes) {
    if (!ctx) return VQ_ERR_INVALID_ARG;
    // Which shapes touch the fixed scratch: the matrix-core kernel of 8-float column blocks (its
    // tables and counters) and the cosine kernels (the centroid norms).  Only they are bound by its
    // size, and only they need the GPU's one array for themselves.
    const bool uses_scratch =
        metric == VQ_COSINE ||
        ((metric == VQ_SQEUCLIDEAN || metric == VQ_EUCLIDEAN) && sd == 8 && ctx->assign_path == 0);
    if (uses_scratch && m > 0 && k > 0 && k <= vq::kMaxK) {
        // the tables of the call must fit: column blocks x centroids padded to 64
        const int64_t cells = (int64_t)m * 64 * ((k + 63) / 64);
        if (m > kNoAllocMaxM || cells > kNoAllocMaxCells)
            return fail(ctx, VQ_ERR_UNSUPPORTED,
                        "vq_assign_noalloc: m * k (k padded to 64) = %lld exceeds the fixed scratch of %d "
                        "(use vq_assign, which may allocate)", (long long)cells, kNoAllocMaxCells);
        if (ctx->device < 0 || ctx->device >= kMaxDevices)
            return fail(ctx, VQ_ERR_UNSUPPORTED, "vq_assign_noalloc: device %d", ctx->device);
        std::lock_guard<std::mutex> lock(g_scratch_mutex);
        vq_ctx *owner = g_scratch_owner[ctx->device];
        if (owner && owner != ctx) {
            const hipError_t busy = hipStreamQuery(owner->stream);
            (void)hipGetLastError();
            if (busy != hipSuccess)
                return fail(ctx, VQ_ERR_UNSUPPORTED,
                            "vq_assign_noalloc: the fixed scratch of GPU %d is in use by another context whose "
                            "stream has not finished (calls that use it must not overlap on one GPU)", ctx->device);
        }
        g_scratch_owner[ctx->device] = ctx;
    }
    // no timing spans (their events are created on demand) and no workspace growth inside the call
    const bool prof = ctx->prof_on;
    ctx->prof_on = false;
    ctx->no_alloc = true;
    const int32_t rc = vqh::assign_codes(ctx, metric, d_x, n, ld, m, sd, k, d_codebooks, d_codes);
    ctx->no_alloc = false;
    ctx->prof_on = prof;
    return rc;
}

int32_t vq_decode_f16(vq_ctx *ctx, const uint8_t *d_codes, int64_t n, int32_t m, int32_t sd, int32_t k,
                      const float *d_codebooks, uint16_t *d_out) {
    return decode_codes<true>(ctx, d_codes, n, m, sd, k, vq::kMaxK, d_codebooks, (void *)d_out);
}

int32_t vq_decode_f32(vq_ctx *ctx, const uint8_t *d_codes, int64_t n, int32_t m, int32_t sd, int32_t k,
                      const float *d_codebooks, float *d_out) {
    return decode_codes<false>(ctx, d_codes, n, m, sd, k, vq::kMaxK, d_codebooks, (void *)d_out);
}

int32_t vq_decode_f16_u16(vq_ctx *ctx, const uint16_t *d_codes, int64_t n, int32_t m, int32_t sd, int32_t k,
                          const float *d_codebooks, uint16_t *d_out) {
    return decode_codes<true>(ctx, d_codes, n, m, sd, k, 65536, d_codebooks, (void *)d_out);
}

int32_t vq_decode_f32_u16(vq_ctx *ctx, const uint16_t *d_codes, int64_t n, int32_t m, int32_t sd, int32_t k,
                          const float *d_codebooks, float *d_out) {
    return decode_codes<false>(ctx, d_codes, n, m, sd, k, 65536, d_codebooks, (void *)d_out);
}

}  // extern "C"

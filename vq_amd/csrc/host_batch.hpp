// Moving rows between the caller's pageable memory and the GPU: a crew of copying threads that the
// context keeps, staged copies in one direction, and batches of host rows through a computation with
// upload, kernels and download of successive chunks side by side.
//
// What bounds it: the host link (about 56 GB/s per direction from page-locked memory) and the copies
// between pageable and page-locked memory, 20-30 GB/s for the caller's thread alone.
#pragma once
#include <hip/hip_runtime.h>

#include <algorithm>
#include <atomic>
#include <condition_variable>
#include <cstring>
#include <functional>
#include <mutex>
#include <thread>
#include <vector>

#include "ctx.hpp"

namespace vqh {

// Threads that sleep between calls; at most one call at a time uses them (a context is not re-entrant).
class CopyCrew {
public:
    ~CopyCrew() {
        {
            std::lock_guard<std::mutex> lock(mutex_);
            stop_ = true;
        }
        wake_.notify_all();
        for (auto &t : threads_) t.join();
    }
    // Wakes up to `count` threads on body(); fewer where the system gives no more.
    void start(int count, const std::function<void()> *body) {
        std::lock_guard<std::mutex> lock(mutex_);
        try {
            while ((int)threads_.size() < count) threads_.emplace_back([this] { loop(); });
        } catch (const std::exception &) {  // the caller copies alone, or with the threads there are
        }
        places_ = count;
        body_ = body;
        wake_.notify_all();
    }
    // Returns once no thread runs body() any more; the body has to know that its work is done.
    void finish() {
        std::unique_lock<std::mutex> lock(mutex_);
        body_ = nullptr;
        idle_.wait(lock, [this] { return running_ == 0; });
    }

private:
    void loop() {
        std::unique_lock<std::mutex> lock(mutex_);
        for (;;) {
            wake_.wait(lock, [this] { return stop_ || (body_ && places_ > 0); });
            if (stop_) return;
            const std::function<void()> *body = body_;
            --places_;
            ++running_;
            lock.unlock();
            (*body)();
            lock.lock();
            if (--running_ == 0) idle_.notify_all();
        }
    }
    std::mutex mutex_;
    std::condition_variable wake_, idle_;
    std::vector<std::thread> threads_;
    const std::function<void()> *body_ = nullptr;
    int places_ = 0, running_ = 0;
    bool stop_ = false;
};

// Pieces of an array, handed out in order up to a moving limit.
struct PieceQueue {
    std::atomic<size_t> next{0}, limit{0};
    bool claim(size_t &piece) {
        size_t p = next.load(std::memory_order_relaxed);
        while (p < limit.load(std::memory_order_acquire))
            if (next.compare_exchange_weak(p, p + 1, std::memory_order_acq_rel)) {
                piece = p;
                return true;
            }
        return false;
    }
};

// One array of `total` bytes in chunks of `chunk` bytes, each copied in pieces of `piece` bytes.
struct Chunks {
    size_t total, chunk, piece, count, per_chunk;
    std::vector<std::atomic<uint32_t>> done;  // pieces copied, per chunk
    Chunks(size_t total_, size_t chunk_, size_t piece_)
        : total(total_), chunk(chunk_), piece(piece_), count((total_ + chunk_ - 1) / chunk_),
          per_chunk((chunk_ + piece_ - 1) / piece_), done(count) {
        for (auto &d : done) d.store(0, std::memory_order_relaxed);
    }
    size_t bytes(size_t c) const { return std::min(chunk, total - c * chunk); }
    bool complete(size_t c) const { return done[c].load(std::memory_order_acquire) == per_chunk; }
    // Piece p between the caller's array and the staging buffer of its chunk.
    template <class Slot>
    void copy(size_t p, char *user, const Slot &slot, bool to_slot) {
        const size_t c = p / per_chunk, lo = std::min(bytes(c), (p % per_chunk) * piece), hi = std::min(bytes(c), lo + piece);
        char *u = user + c * chunk + lo, *s = slot(c) + lo;
        if (hi > lo) memcpy(to_slot ? s : u, to_slot ? u : s, hi - lo);
        done[c].fetch_add(1, std::memory_order_release);
    }
};

// How many threads help the caller with `bytes`.  None below 64 MB: lines that other processors have read
// or written have to be taken back from their caches when the caller's thread next touches them, which
// costs it about what the help saves (50,000 x 128 rows quantized: 1.62 -> 0.94 ms, the caller's next write of
// its rows 0.60 -> 1.19 ms; 10,000: 0.32 -> 0.36 and 0.07 -> 0.31).  Help with the results alone does not pay
// either (50,000 rows: 1.62 ms, with three threads 1.49, with seven 1.69; 80,000: 2.6, 3.1, 2.6).  Larger arrays
// do not stay in caches.
inline int crew_for(size_t bytes) {
    const unsigned hw = std::thread::hardware_concurrency();
    return bytes < (64u << 20) ? 0 : (int)std::min<unsigned>(7u, hw > 2 ? hw / 2 - 1 : 0u);
}

CopyCrew &crew(vq_ctx *ctx);

// Copies `bytes` between pageable host memory and the GPU through page-locked staging buffers: the
// crew fills (or empties) the chunk behind the one that the copy engine moves.  Synchronises.
int32_t staged_copy(vq_ctx *ctx, void *d, void *h, size_t bytes, bool upload);

// A caller's array of results: bytes per row, null if it is not asked for.
struct HostOut {
    void *h;
    size_t row;
};
// n host rows of row_in bytes through run(d_x, rows, d_out0, d_out1), which enqueues the computation of a
// chunk on the context's stream and writes every row of both outputs; chunks of about chunk_bytes.
// direct (run's kernels read each row once or twice): a few rows are read from and written to page-locked
// memory in place.  Synchronises.
using HostRun = std::function<int32_t(const float *, int64_t, void *, void *)>;
int32_t host_batch(vq_ctx *ctx, const float *h_x, int64_t n, size_t row_in, const HostOut (&outs)[2], size_t chunk_bytes,
                   bool direct, const HostRun &run);

}  // namespace vqh

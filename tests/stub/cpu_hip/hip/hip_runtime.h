// A stand-in for the parts of the HIP runtime that vq_api_host.hip uses, for ONE purpose: running the
// library's host-side copies and batches under the thread and address sanitizers on machines without a GPU.
// Test infrastructure only.  Two devices; "device" memory is host memory of exactly the size asked for;
// a stream is a thread that works off a queue, so copies and kernels are as asynchronous as on a GPU and a
// missing wait is a data race that the thread sanitizer reports.  As in HIP, streams and events belong to
// the device that was current at their creation, and an event is recorded on streams of its device only.
#pragma once
#include <atomic>
#include <condition_variable>
#include <cstddef>
#include <cstdint>
#include <cstdlib>
#include <cstring>
#include <deque>
#include <functional>
#include <mutex>
#include <set>
#include <thread>

enum hipError_t {
    hipSuccess = 0,
    hipErrorInvalidValue = 1,
    hipErrorOutOfMemory = 2,
    hipErrorInvalidHandle = 400,
    hipErrorNotReady = 600,
    hipErrorUnknown = 999
};
enum hipMemcpyKind { hipMemcpyHostToDevice = 1, hipMemcpyDeviceToHost = 2, hipMemcpyDeviceToDevice = 3 };
enum hipMemoryType { hipMemoryTypeUnregistered = 0, hipMemoryTypeHost = 1, hipMemoryTypeDevice = 2 };
struct hipPointerAttribute_t {
    hipMemoryType type;
};
constexpr unsigned hipStreamNonBlocking = 1, hipEventDisableTiming = 2, hipHostMallocDefault = 0;

struct dim3 {
    unsigned x, y, z;
    dim3(unsigned x_ = 1, unsigned y_ = 1, unsigned z_ = 1) : x(x_), y(y_), z(z_) {}
};
struct alignas(16) uint4 {
    uint32_t x, y, z, w;
};
#define __global__
#define __launch_bounds__(n)

namespace cpu_hip {

constexpr int kDevices = 2;
inline thread_local int current = 0;
inline thread_local dim3 grid_dim, block_idx, thread_idx;
inline std::atomic<int> copies{0};        // hipMemcpyAsync calls so far
inline std::atomic<int> fail_copy_at{0};  // the number of the call that is to fail (0: none)

struct Stream {
    int device;
    std::mutex mutex;
    std::condition_variable wake, idle;
    std::deque<std::function<void()>> queue;
    bool busy = false, stop = false;
    std::thread worker;
    explicit Stream(int d) : device(d), worker([this] { loop(); }) {}
    ~Stream() {
        wait();
        {
            std::lock_guard<std::mutex> lock(mutex);
            stop = true;
        }
        wake.notify_all();
        worker.join();
    }
    void push(std::function<void()> f) {
        std::lock_guard<std::mutex> lock(mutex);
        queue.push_back(std::move(f));
        wake.notify_one();
    }
    void wait() {
        std::unique_lock<std::mutex> lock(mutex);
        idle.wait(lock, [this] { return queue.empty() && !busy; });
    }

private:
    void loop() {
        std::unique_lock<std::mutex> lock(mutex);
        for (;;) {
            wake.wait(lock, [this] { return stop || !queue.empty(); });
            if (queue.empty()) return;
            std::function<void()> f = std::move(queue.front());
            queue.pop_front();
            busy = true;
            lock.unlock();
            std::this_thread::yield();
            f();
            f = nullptr;
            lock.lock();
            busy = false;
            if (queue.empty()) idle.notify_all();
        }
    }
};

struct Event {
    int device;
    std::atomic<uint64_t> recorded{0}, reached{0};
    explicit Event(int d) : device(d) {}
};

inline std::mutex locked_mutex;
inline std::set<void *> locked;  // page-locked allocations

template <class F>
void launch(Stream *s, dim3 grid, dim3 block, F body) {
    s->push([=] {
        grid_dim = grid;
        for (unsigned b = 0; b < grid.x; ++b)
            for (unsigned t = 0; t < block.x; ++t) {
                block_idx = dim3(b);
                thread_idx = dim3(t);
                body();
            }
    });
}

}  // namespace cpu_hip

#define gridDim cpu_hip::grid_dim
#define blockIdx cpu_hip::block_idx
#define threadIdx cpu_hip::thread_idx
#define hipLaunchKernelGGL(kern, grid, block, lds, stream, ...) \
    cpu_hip::launch(stream, grid, block, [=] { kern(__VA_ARGS__); })

using hipStream_t = cpu_hip::Stream *;
using hipEvent_t = cpu_hip::Event *;

inline const char *hipGetErrorString(hipError_t e) { return e == hipSuccess ? "no error" : "error"; }
inline hipError_t hipGetLastError() { return hipSuccess; }
inline hipError_t hipSetDevice(int d) {
    if (d < 0 || d >= cpu_hip::kDevices) return hipErrorInvalidValue;
    cpu_hip::current = d;
    return hipSuccess;
}
inline hipError_t hipStreamCreateWithFlags(hipStream_t *s, unsigned) {
    *s = new cpu_hip::Stream(cpu_hip::current);
    return hipSuccess;
}
inline hipError_t hipStreamDestroy(hipStream_t s) {
    delete s;
    return hipSuccess;
}
inline hipError_t hipStreamSynchronize(hipStream_t s) {
    s->wait();
    return hipSuccess;
}
inline hipError_t hipEventCreateWithFlags(hipEvent_t *e, unsigned) {
    *e = new cpu_hip::Event(cpu_hip::current);
    return hipSuccess;
}
inline hipError_t hipEventCreate(hipEvent_t *e) { return hipEventCreateWithFlags(e, 0); }
inline hipError_t hipEventDestroy(hipEvent_t e) {
    delete e;
    return hipSuccess;
}
inline hipError_t hipEventRecord(hipEvent_t e, hipStream_t s) {
    if (e->device != s->device) return hipErrorInvalidHandle;
    const uint64_t at = e->recorded.fetch_add(1) + 1;
    s->push([=] { e->reached.store(at, std::memory_order_release); });
    return hipSuccess;
}
inline hipError_t hipEventQuery(hipEvent_t e) {
    return e->reached.load(std::memory_order_acquire) == e->recorded.load() ? hipSuccess : hipErrorNotReady;
}
inline hipError_t hipStreamWaitEvent(hipStream_t s, hipEvent_t e, unsigned) {
    const uint64_t at = e->recorded.load();
    s->push([=] {
        while (e->reached.load(std::memory_order_acquire) < at) std::this_thread::yield();
    });
    return hipSuccess;
}
inline hipError_t hipEventElapsedTime(float *ms, hipEvent_t, hipEvent_t) {
    *ms = 0.0f;
    return hipSuccess;
}
inline hipError_t hipMemcpyAsync(void *dst, const void *src, size_t bytes, hipMemcpyKind, hipStream_t s) {
    if (++cpu_hip::copies == cpu_hip::fail_copy_at.load()) return hipErrorUnknown;
    s->push([=] { memcpy(dst, src, bytes); });
    return hipSuccess;
}
inline hipError_t hipMalloc(void **p, size_t bytes) {
    *p = std::aligned_alloc(256, (bytes + 255) & ~(size_t)255);
    return *p ? hipSuccess : hipErrorOutOfMemory;
}
inline hipError_t hipFree(void *p) {
    std::free(p);
    return hipSuccess;
}
inline hipError_t hipHostMalloc(void **p, size_t bytes, unsigned) {
    if (hipMalloc(p, bytes) != hipSuccess) return hipErrorOutOfMemory;
    std::lock_guard<std::mutex> lock(cpu_hip::locked_mutex);
    cpu_hip::locked.insert(*p);
    return hipSuccess;
}
inline hipError_t hipHostFree(void *p) {
    std::lock_guard<std::mutex> lock(cpu_hip::locked_mutex);
    cpu_hip::locked.erase(p);
    std::free(p);
    return hipSuccess;
}
inline hipError_t hipPointerGetAttributes(hipPointerAttribute_t *a, const void *p) {
    std::lock_guard<std::mutex> lock(cpu_hip::locked_mutex);
    if (!cpu_hip::locked.count(const_cast<void *>(p))) return hipErrorInvalidValue;
    a->type = hipMemoryTypeHost;
    return hipSuccess;
}

// A HIP runtime on the host, as far as nuc_transfer.hip uses it, for tests of
// its threads, its locks and its ordering without a GPU.  Streams run their work
// in order on a thread each.  Pinned memory without hipHostMallocCoherent shows a
// kernel's stores to the host only after a release at system scope, the least
// that HIP promises: a stream synchronisation, or an event that asks for it.
#pragma once
#include <stddef.h>
#include <stdint.h>

#include <condition_variable>
#include <cstring>
#include <deque>
#include <functional>
#include <map>
#include <memory>
#include <mutex>
#include <thread>
#include <vector>

enum hipError_t { hipSuccess = 0, hipErrorInvalidValue = 1, hipErrorOutOfMemory = 2 };
enum hipMemcpyKind { hipMemcpyHostToDevice = 1, hipMemcpyDeviceToHost = 2 };
enum hipMemoryType { hipMemoryTypeUnregistered = 0, hipMemoryTypeHost = 1, hipMemoryTypeDevice = 2 };
struct hipPointerAttribute_t { hipMemoryType type; };
constexpr unsigned hipHostMallocDefault = 0x0, hipHostMallocPortable = 0x1, hipHostMallocCoherent = 0x40000000;
constexpr unsigned hipEventDisableTiming = 0x2, hipEventReleaseToSystem = 0x80000000;

struct dim3 {
    unsigned x, y, z;
    dim3(unsigned x_ = 1, unsigned y_ = 1, unsigned z_ = 1) : x(x_), y(y_), z(z_) {}
};
inline thread_local dim3 blockIdx, blockDim, gridDim, threadIdx;
#define __global__
#define __device__
#define __launch_bounds__(...)

namespace hosthip {

inline thread_local int device = 0;     // current device of the calling thread
inline int refuse_pinned = 0;           // hipHostMalloc fails while set
inline thread_local int inside = 0;     // calls of this runtime on the thread's stack
struct Inside { Inside() { inside++; } ~Inside() { inside--; } };
inline int staged_kernels = 0, plain_copies = 0, pinned_copies = 0;
inline std::mutex mu;                   // the maps and counters below and above
struct Pinned { size_t bytes; bool coherent; };
inline std::map<char *, Pinned> pinned;

inline std::map<char *, Pinned>::iterator pinned_of(const void *p)
{
    char *c = static_cast<char *>(const_cast<void *>(p));
    auto it = pinned.upper_bound(c);
    if (it == pinned.begin()) return pinned.end();
    --it;
    return c < it->first + it->second.bytes ? it : pinned.end();
}

struct Stream {
    int dev;
    std::mutex m;
    std::condition_variable cv;
    std::deque<std::function<void()>> q;
    bool busy = false, stop = false;
    std::vector<std::pair<char *, std::vector<char>>> unreleased;   // stores the host does not see yet
    std::thread th;
    explicit Stream(int d) : dev(d), th([this] { run(); }) {}
    ~Stream()
    {
        { std::lock_guard<std::mutex> l(m); stop = true; }
        cv.notify_all();
        th.join();
    }
    void run()
    {
        std::unique_lock<std::mutex> l(m);
        for (;;) {
            cv.wait(l, [this] { return stop || !q.empty(); });
            if (q.empty()) return;
            auto f = std::move(q.front());
            q.pop_front();
            busy = true;
            l.unlock();
            f();
            l.lock();
            busy = false;
            cv.notify_all();
        }
    }
    void put(std::function<void()> f)
    {
        { std::lock_guard<std::mutex> l(m); q.push_back(std::move(f)); }
        cv.notify_all();
    }
    void release()
    {
        for (auto &u : unreleased) std::memcpy(u.first, u.second.data(), u.second.size());
        unreleased.clear();
    }
    void sync()
    {
        put([this] { release(); });
        std::unique_lock<std::mutex> l(m);
        cv.wait(l, [this] { return q.empty() && !busy; });
    }
};

struct Event {
    unsigned flags;
    std::mutex m;
    std::condition_variable cv;
    int recorded = 0, reached = 0;
};

}  // namespace hosthip

using hipStream_t = hosthip::Stream *;
using hipEvent_t = std::shared_ptr<hosthip::Event>;

inline hipError_t hipGetLastError() { return hipSuccess; }
inline hipError_t hipGetDevice(int *d) { *d = hosthip::device; return hipSuccess; }
inline hipError_t hipSetDevice(int d) { hosthip::device = d; return hipSuccess; }
inline hipError_t hipStreamGetDevice(hipStream_t s, int *d) { *d = s->dev; return hipSuccess; }
inline hipError_t hipStreamSynchronize(hipStream_t s) { hosthip::Inside in; s->sync(); return hipSuccess; }

inline hipError_t hipHostMalloc(void **p, size_t n, unsigned flags)
{
    hosthip::Inside in;
    std::lock_guard<std::mutex> l(hosthip::mu);
    if (hosthip::refuse_pinned) return hipErrorOutOfMemory;
    char *c = new char[n];
    std::memset(c, 0x5A, n);
    hosthip::pinned[c] = {n, (flags & hipHostMallocCoherent) != 0 || flags == hipHostMallocDefault};
    *p = c;
    return hipSuccess;
}
inline hipError_t hipHostFree(void *p)
{
    hosthip::Inside in;
    std::lock_guard<std::mutex> l(hosthip::mu);
    hosthip::pinned.erase(static_cast<char *>(p));
    delete[] static_cast<char *>(p);
    return hipSuccess;
}
inline hipError_t hipPointerGetAttributes(hipPointerAttribute_t *a, const void *p)
{
    std::lock_guard<std::mutex> l(hosthip::mu);
    if (hosthip::pinned_of(p) == hosthip::pinned.end()) return hipErrorInvalidValue;
    a->type = hipMemoryTypeHost;
    return hipSuccess;
}

inline hipError_t hipEventCreateWithFlags(hipEvent_t *e, unsigned flags)
{
    hosthip::Inside in;
    *e = std::make_shared<hosthip::Event>();
    (*e)->flags = flags;
    return hipSuccess;
}
inline hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
inline hipError_t hipEventRecord(hipEvent_t e, hipStream_t s)
{
    hosthip::Inside in;
    int n;
    { std::lock_guard<std::mutex> l(e->m); n = ++e->recorded; }
    s->put([e, s, n] {
        if (e->flags & hipEventReleaseToSystem) s->release();
        { std::lock_guard<std::mutex> l(e->m); e->reached = n; }
        e->cv.notify_all();
    });
    return hipSuccess;
}
inline hipError_t hipEventSynchronize(hipEvent_t e)
{
    std::unique_lock<std::mutex> l(e->m);
    e->cv.wait(l, [&] { return e->reached == e->recorded; });
    return hipSuccess;
}
inline hipError_t hipMemcpyAsync(void *d, const void *s, size_t n, hipMemcpyKind kind, hipStream_t st)
{
    hosthip::Inside in;
    {
        std::lock_guard<std::mutex> l(hosthip::mu);
        const void *host = kind == hipMemcpyHostToDevice ? s : d;
        (hosthip::pinned_of(host) == hosthip::pinned.end() ? hosthip::plain_copies : hosthip::pinned_copies)++;
    }
    st->put([=] { std::memcpy(d, s, n); });
    return hipSuccess;
}

// a kernel (source, destination, count of V): its stores to non-coherent pinned
// memory wait for the stream's next system-scope release
template <typename V>
void launch(void (*k)(const V *, V *, size_t), dim3 grid, dim3 block, hipStream_t s, const V *src, V *dst, size_t n)
{
    hosthip::Inside in;
    s->put([=] {
        char *const d = reinterpret_cast<char *>(dst);
        const size_t bytes = n * sizeof(V);
        bool hidden;
        {
            std::lock_guard<std::mutex> l(hosthip::mu);
            auto it = hosthip::pinned_of(d);
            hidden = it != hosthip::pinned.end() && !it->second.coherent;
            hosthip::staged_kernels++;
        }
        std::vector<char> before;
        if (hidden) before.assign(d, d + bytes);
        gridDim = grid;
        blockDim = block;
        for (blockIdx.x = 0; blockIdx.x < grid.x; blockIdx.x++)
            for (threadIdx.x = 0; threadIdx.x < block.x; threadIdx.x++) k(src, dst, n);
        if (hidden) {
            s->unreleased.emplace_back(d, std::vector<char>(d, d + bytes));
            std::memcpy(d, before.data(), bytes);
        }
    });
}
#define hipLaunchKernelGGL(kernel, grid, block, shared, stream, ...) launch(kernel, grid, block, stream, __VA_ARGS__)

// nuc_transfer.hip -- copies of states and fields between pageable host arrays
// and the device through pinned staging memory, by several host threads.
//
// hipMemcpyAsync on a pageable array stages it through the runtime's own
// pinned buffers on the calling thread, which pays for the memory copy and, on
// a fresh array, for its page faults.  Here each of THREADS workers owns two
// pinned slots and every THREADS-th chunk of the array: while one slot's chunk
// is on the link, the worker copies (and faults in) the other's.
// Measured on a fresh 671 MB array (256^3): up 22.5 -> 14.5 ms (46 GB/s), down
// 63.9 -> 14.6 ms (46 GB/s); 5.4 GB: up 193 -> 114, down 582 -> 110 ms; 35 MB:
// up 1.14 -> 0.94, down 3.6 -> 1.3 ms.  The link carries about 50 GB/s.
#include "nuc_transfer.h"

#include <algorithm>
#include <atomic>
#include <cstdint>
#include <cstring>
#include <exception>
#include <mutex>
#include <thread>
#include <utility>

namespace nuctransfer {
namespace {

constexpr int THREADS = 8;
constexpr size_t CHUNK = size_t(4) << 20;
constexpr int OUT_BLOCKS = 16;         // fill the link (16 to 256 measured alike)
// Smaller arrays take the runtime's path: the workers' start and the larger
// chunks cost more than they save (10 MB up 0.30 ms against 0.6-3.9 staged,
// down 0.79 against 0.63; 35 MB up 1.14 against 0.94).
constexpr size_t MIN_UP = size_t(16) << 20, MIN_DOWN = size_t(8) << 20;

// What staging a copy saves, us, by the measurements above and (whole passes of
// upload, step and download) 17 MB down 0.5 ms, 10 MB 0.2 ms.
size_t saving(size_t bytes, bool up) { return (bytes >> 20) * (up ? 10 : bytes >= (size_t(32) << 20) ? 70 : 20); }
// Pinning a slot and giving it back takes 0.4-0.6 ms (all of them 6-10): as many as
// the array has chunks are pinned, and only once the copies have lost more than their
// price, which a 256^3 state does in its first way down, a 96^3 one in its third pass
// and a 64^3 one (three slots) in its twelfth.  All pinned at the first 64 MiB they made
// contexts that live for a few copies slower than the runtime's own (96^3, created,
// stepped once and destroyed: 8.4 -> 15.2 ms; 76^3 with four passes 11 -> 18).
constexpr size_t PIN_AFTER = 800;      // us a slot

std::mutex g_users_mu;                 // the user count
int g_users = 0;
// The staging memory and what follows.  Held while a copy is staged, but neither
// by callers that only come or go nor while a copy waits for its stream's earlier
// work, so that contexts are created and destroyed, and others copy, beside one
// that downloads behind queued steps.  Taken after g_users_mu where both are.
std::mutex g_stage_mu;
// Slots of CHUNK bytes, the first g_slots of them pinned (all: 64 MiB), in g_blocks
// blocks; worker w's are w and THREADS + w.  Coherent: a worker reads a slot once the
// event behind its kernel is reached, and only coherent memory is promised to show
// a kernel's stores by then (other pinned memory: after a release at system scope,
// which an event need not be).  As fast: 256^3 down 14.8 and 14.7 ms, up 14.6 and
// 14.5.
char *g_slot[2 * THREADS], *g_block[2 * THREADS];
int g_slots = 0, g_blocks = 0;
size_t g_lost = 0;                     // us that copies lost by not being staged since slots were last pinned or given back

// A chunk into a pinned slot by stores over the link.  hipMemcpyAsync down
// followed by an event costs 130 us a copy here whatever its size (4 MiB
// chunks 18 GB/s), a kernel's event does not.
template <typename V>
__global__ __launch_bounds__(256) void k_out(const V *src, V *dst, size_t n)
{
    for (size_t i = (size_t)blockIdx.x * 256 + threadIdx.x; i < n; i += (size_t)gridDim.x * 256)
        __builtin_nontemporal_store(src[i], dst + i);
}
using v2d = __attribute__((ext_vector_type(2))) double;

// one worker's chunks w, w + THREADS, ...; the first error stops the others
void work(int w, char *host, char *dev, size_t bytes, bool up, hipStream_t s, int device, std::atomic<int> *err)
{
    char *const slot[2] = {g_slot[w], g_slot[THREADS + w]};
    hipEvent_t ev[2] = {nullptr, nullptr};
    hipError_t e = hipSetDevice(device);
    for (int k = 0; k < 2 && e == hipSuccess; k++) e = hipEventCreateWithFlags(&ev[k], hipEventDisableTiming);
    const size_t n = (bytes + CHUNK - 1) / CHUNK;
    auto len = [&](size_t c) { return std::min(CHUNK, bytes - c * CHUNK); };
    auto fetch = [&](size_t c, int k) {   // down: chunk c onto slot k
        const char *src = dev + c * CHUNK;
        if (reinterpret_cast<uintptr_t>(src) % 16 == 0 && len(c) % 16 == 0)
            hipLaunchKernelGGL(k_out<v2d>, dim3(OUT_BLOCKS), dim3(256), 0, s, reinterpret_cast<const v2d *>(src),
                               reinterpret_cast<v2d *>(slot[k]), len(c) / 16);
        else
            hipLaunchKernelGGL(k_out<double>, dim3(OUT_BLOCKS), dim3(256), 0, s, reinterpret_cast<const double *>(src),
                               reinterpret_cast<double *>(slot[k]), len(c) / 8);
        hipError_t r = hipGetLastError();
        return r == hipSuccess ? hipEventRecord(ev[k], s) : r;
    };
    if (!up && e == hipSuccess && (size_t)w < n) e = fetch(w, 0);
    int k = 0;
    for (size_t c = w; c < n && e == hipSuccess && err->load(std::memory_order_relaxed) == hipSuccess; c += THREADS, k ^= 1) {
        if (up) {
            if (c >= (size_t)w + 2 * THREADS) e = hipEventSynchronize(ev[k]);   // the slot's earlier chunk is out
            if (e != hipSuccess) break;
            std::memcpy(slot[k], host + c * CHUNK, len(c));
            e = hipMemcpyAsync(dev + c * CHUNK, slot[k], len(c), hipMemcpyHostToDevice, s);
            if (e == hipSuccess) e = hipEventRecord(ev[k], s);
        } else {
            if (c + THREADS < n) e = fetch(c + THREADS, k ^ 1);
            if (e == hipSuccess) e = hipEventSynchronize(ev[k]);
            if (e == hipSuccess) std::memcpy(host + c * CHUNK, slot[k], len(c));
        }
    }
    if (e != hipSuccess) {
        int none = hipSuccess;
        err->compare_exchange_strong(none, (int)e);
    }
    for (int i = 0; i < 2; i++)
        if (ev[i]) (void)hipEventDestroy(ev[i]);
}

// the first n slots pinned, the missing ones in one block (each by itself: twice the time)
void pin(int n)
{
    char *block = nullptr;
    if (hipHostMalloc((void **)&block, (n - g_slots) * CHUNK, hipHostMallocPortable | hipHostMallocCoherent) != hipSuccess) {
        (void)hipGetLastError();
        return;
    }
    g_block[g_blocks++] = block;
    for (; g_slots < n; g_slots++, block += CHUNK) g_slot[g_slots] = block;
}

// whether the runtime knows the pointer (pinned, managed or device memory):
// those are copied without staging
bool known(const void *p)
{
    hipPointerAttribute_t a;
    std::memset(&a, 0, sizeof(a));
    const hipError_t e = hipPointerGetAttributes(&a, p);
    if (e != hipSuccess) {
        (void)hipGetLastError();   // an ordinary pageable pointer
        return false;
    }
    return a.type != hipMemoryTypeUnregistered;
}

}  // namespace

hipError_t copy(void *dst, const void *src, size_t bytes, hipMemcpyKind kind, hipStream_t s)
{
    const bool up = kind == hipMemcpyHostToDevice;
    const void *host = up ? src : dst;
    if (bytes >= (up ? MIN_UP : MIN_DOWN) && bytes % 8 == 0 && !known(host)) {
        const hipError_t earlier = hipStreamSynchronize(s);   // before the staging memory is taken
        if (earlier != hipSuccess) return earlier;
        // one staged copy at a time; another thread's takes the plain path meanwhile
        std::unique_lock<std::mutex> lk(g_stage_mu, std::try_to_lock);
        if (lk.owns_lock()) {
            const int need = (int)std::min<size_t>(2 * THREADS, (bytes + CHUNK - 1) / CHUNK);
            if (g_slots < need) {
                g_lost += saving(bytes, up);
                if (g_lost >= PIN_AFTER * (need - g_slots)) {
                    pin(need);
                    g_lost = 0;
                }
            }
            int device = 0, callers = 0;
            if (g_slots >= need && hipStreamGetDevice(s, &device) == hipSuccess && hipGetDevice(&callers) == hipSuccess) {
                std::atomic<int> err{hipSuccess};
                char *h = static_cast<char *>(const_cast<void *>(host)), *d = static_cast<char *>(up ? dst : const_cast<void *>(src));
                std::thread th[THREADS];
                int started = 0;
                try {
                    for (; started < THREADS - 1; started++)
                        th[started] = std::thread(work, started + 1, h, d, bytes, up, s, device, &err);
                } catch (const std::exception &) {
                    // no more threads, or no memory to start one: the calling one does the rest
                }
                work(0, h, d, bytes, up, s, device, &err);
                for (int w = started + 1; w < THREADS; w++) work(w, h, d, bytes, up, s, device, &err);
                for (int i = 0; i < started; i++) th[i].join();
                if (callers != device) (void)hipSetDevice(callers);   // work() has set the stream's
                // the slots are free for the next copy only when every copy has left them
                const hipError_t e = hipStreamSynchronize(s);
                return err.load() != hipSuccess ? (hipError_t)err.load() : e;
            }
        }
    }
    const hipError_t e = hipMemcpyAsync(dst, src, bytes, kind, s);
    return e == hipSuccess ? hipStreamSynchronize(s) : e;
}

void retain()
{
    std::lock_guard<std::mutex> lk(g_users_mu);
    g_users++;
}

void release()
{
    char *gone[2 * THREADS];
    int n = 0;
    {
        std::lock_guard<std::mutex> lk(g_users_mu);
        if (--g_users == 0) {
            std::lock_guard<std::mutex> st(g_stage_mu);   // free: no user is left to copy
            std::swap(n, g_blocks);
            std::copy(g_block, g_block + n, gone);
            g_slots = 0;
            g_lost = 0;
        }
    }
    for (int i = 0; i < n; i++) (void)hipHostFree(gone[i]);
}

}  // namespace nuctransfer

// nuc_transfer.hip over a HIP runtime on the host (host_hip): what its copies
// promise about the bytes, the threads beside them and the calling thread.
#include "nuc_transfer.hip"

#include <chrono>
#include <cstdio>
#include <cstdlib>
#include <future>
#include <string>

static int failed = 0;
#define CHECK(c, ...) do { if (!(c)) { failed++; std::printf("line %d: %s: ", __LINE__, #c); std::printf(__VA_ARGS__); std::printf("\n"); } } while (0)

static std::vector<double> values(size_t n, unsigned seed)
{
    std::vector<double> v(n);
    uint64_t x = seed * 2654435761u + 1;
    for (double &d : v) { x = x * 6364136223846793005ull + 1442695040888963407ull; d = double(x >> 11); }
    return v;
}

// past the copies after which the staging memory is pinned
static void warm(hosthip::Stream &s)
{
    std::vector<double> a(size_t(9) << 20), d(a.size());
    for (int i = 0; i < 4; i++) nuctransfer::copy(d.data(), a.data(), 8 * a.size(), hipMemcpyDeviceToHost, &s);
    hosthip::staged_kernels = hosthip::plain_copies = hosthip::pinned_copies = 0;
}

// Bytes both ways at sizes around the limits and the chunks; `off` values of the
// device array are skipped, so that its chunks begin 8 bytes off 16
static void bytes()
{
    hosthip::Stream s(0);
    nuctransfer::retain();
    warm(s);
    const size_t MB = size_t(1) << 20;
    const size_t sizes[] = {8 * MB - 8, 8 * MB, 8 * MB + 8, 16 * MB - 8, 16 * MB, 16 * MB + 8, 20 * MB, 32 * MB,
                            32 * MB + 8, 36 * MB - 16, 64 * MB + 24, 69 * MB + 8};
    for (size_t n8 : sizes)
        for (size_t off : {0, 1}) {
            const size_t n = n8 / 8;
            std::vector<double> h = values(n, unsigned(n + off)), d(n + off + 2, -1.0), back(n + 2, -2.0);
            hosthip::staged_kernels = hosthip::plain_copies = hosthip::pinned_copies = 0;
            CHECK(nuctransfer::copy(d.data() + off, h.data(), n8, hipMemcpyHostToDevice, &s) == hipSuccess, "up");
            CHECK(std::memcmp(d.data() + off, h.data(), n8) == 0 && d[n + off] == -1.0, "%zu bytes up", n8);
            CHECK((hosthip::pinned_copies > 0) == (n8 >= 16 * MB), "%zu bytes up: %d staged", n8, hosthip::pinned_copies);
            for (size_t i = 0; i < n; i++) h[i] = d[off + i] = h[i] + 1.0;   // other bytes than the slots still hold
            CHECK(nuctransfer::copy(back.data(), d.data() + off, n8, hipMemcpyDeviceToHost, &s) == hipSuccess, "down");
            CHECK(std::memcmp(back.data(), h.data(), n8) == 0 && back[n] == -2.0, "%zu bytes down, offset %zu", n8, off);
            CHECK((hosthip::staged_kernels > 0) == (n8 >= 8 * MB), "%zu bytes down: %d staged", n8, hosthip::staged_kernels);
        }
    // memory the runtime knows, and sizes that are no whole number of doubles, are not staged
    void *p = nullptr;
    CHECK(hipHostMalloc(&p, 32 * MB, hipHostMallocDefault) == hipSuccess, "pinned");
    std::vector<double> d(4 * MB);
    hosthip::staged_kernels = hosthip::plain_copies = hosthip::pinned_copies = 0;
    CHECK(nuctransfer::copy(p, d.data(), 32 * MB, hipMemcpyDeviceToHost, &s) == hipSuccess, "down");
    CHECK(hosthip::staged_kernels == 0 && hosthip::pinned_copies == 1, "a pinned array is copied as it is");
    std::vector<char> odd(32 * MB);
    CHECK(nuctransfer::copy(odd.data(), d.data(), 32 * MB - 3, hipMemcpyDeviceToHost, &s) == hipSuccess, "down");
    CHECK(hosthip::staged_kernels == 0 && hosthip::plain_copies == 1, "%d", hosthip::staged_kernels);
    hipHostFree(p);
    nuctransfer::release();
    CHECK(hosthip::pinned.empty(), "the staging memory is given back");
    // where no memory can be pinned the runtime copies
    nuctransfer::retain();
    hosthip::refuse_pinned = 1;
    std::vector<double> h = values(size_t(10) * MB, 7), e(h.size());
    for (int i = 0; i < 4; i++)
        CHECK(nuctransfer::copy(e.data(), h.data(), 8 * h.size(), hipMemcpyDeviceToHost, &s) == hipSuccess && e == h, "refused");
    CHECK(hosthip::pinned.empty(), "refused");
    hosthip::refuse_pinned = 0;
    nuctransfer::release();
}

// Slots are pinned once copies have lost 0.8 ms for each that the array needs: on a
// 704 MB array's way down, but not for the few copies of a short-lived context, whose
// sum starts again with the next one; and no more than the array needs
static void pinning()
{
    hosthip::Stream s(0);
    std::vector<double> a(size_t(84) << 20), d(a.size());   // 704 MB
    size_t slots = 0;
    auto passes = [&](size_t bytes, int n) {
        int pinned = 0;
        slots = 0;
        nuctransfer::retain();
        for (int i = 0; i < n; i++) {
            nuctransfer::copy(d.data(), a.data(), bytes, hipMemcpyHostToDevice, &s);
            nuctransfer::copy(a.data(), d.data(), bytes, hipMemcpyDeviceToHost, &s);
            if (!pinned && !hosthip::pinned.empty()) pinned = i + 1;
            slots = 0;
            for (auto &p : hosthip::pinned) slots += p.second.bytes >> 22;
        }
        nuctransfer::release();
        CHECK(hosthip::pinned.empty(), "given back");
        return pinned;
    };
    const size_t c96 = 40 * 96 * 96 * 96, c76 = 40 * 76 * 76 * 76, c64 = 40 * 64 * 64 * 64;
    for (int contexts = 0; contexts < 6; contexts++) CHECK(passes(c96, 2) == 0, "96^3, two passes");
    const int p96 = passes(c96, 6);
    CHECK(p96 == 3 && slots == 9, "96^3: pass %d, %zu slots", p96, slots);
    const int p76 = passes(c76, 20);
    CHECK(p76 >= 7 && p76 <= 12 && slots == 5, "76^3: pass %d, %zu slots", p76, slots);
    const int p64 = passes(c64, 30);
    CHECK(p64 >= 10 && p64 <= 15 && slots == 3, "64^3: pass %d, %zu slots", p64, slots);
    CHECK(passes(8 * a.size(), 1) == 1 && slots == 16, "704 MB: %zu slots", slots);
}

// A copy behind a stream's earlier work: contexts and serving loops come and go
// meanwhile, and another stream's copy is staged
static void locks()
{
    hosthip::Stream a(0), b(0);
    nuctransfer::retain();
    warm(a);
    std::promise<void> gate;
    std::shared_future<void> open = gate.get_future().share();
    a.put([open] { open.wait(); });
    std::vector<double> da = values(size_t(5) << 20, 1), db = values(size_t(5) << 20, 2), ha(da.size()), hb(db.size());
    std::thread ta([&] { nuctransfer::copy(ha.data(), da.data(), 8 * da.size(), hipMemcpyDeviceToHost, &a); });
    std::this_thread::sleep_for(std::chrono::milliseconds(200));   // into its copy
    auto wait = [](std::future<void> &f) { return f.wait_for(std::chrono::seconds(10)) == std::future_status::ready; };
    std::future<void> user = std::async(std::launch::async, [] { nuctransfer::retain(); nuctransfer::release(); });
    CHECK(wait(user), "retain and release wait for another stream's work");
    std::future<void> other = std::async(std::launch::async, [&] {
        nuctransfer::copy(hb.data(), db.data(), 8 * db.size(), hipMemcpyDeviceToHost, &b);
    });
    CHECK(wait(other), "a copy waits for another stream's work");
    CHECK(hosthip::staged_kernels > 0, "the copy beside a waiting one is not staged");
    gate.set_value();
    ta.join();
    user.get();
    other.get();
    CHECK(ha == da && hb == db, "bytes");
    nuctransfer::release();
    CHECK(hosthip::pinned.empty(), "the staging memory is given back");
}

// The calling thread's current device is its own
static void device()
{
    hosthip::Stream s(1);
    nuctransfer::retain();
    warm(s);
    std::vector<double> h = values(size_t(5) << 20, 3), d(h.size()), r(h.size());
    hosthip::device = 0;
    nuctransfer::copy(d.data(), h.data(), 8 * h.size(), hipMemcpyHostToDevice, &s);
    CHECK(hosthip::device == 0, "device %d after a copy up", hosthip::device);
    hosthip::device = 0;
    nuctransfer::copy(r.data(), d.data(), 8 * d.size(), hipMemcpyDeviceToHost, &s);
    CHECK(hosthip::device == 0, "device %d after a copy down", hosthip::device);
    CHECK(r == h && hosthip::staged_kernels > 0 && hosthip::pinned_copies > 0, "bytes, staged");
    nuctransfer::release();
}

// While set, this thread's allocations outside the runtime fail (a worker
// thread's start among them)
static thread_local bool refuse_new = false;

void *operator new(size_t n)
{
    if (refuse_new && !hosthip::inside) throw std::bad_alloc();
    if (void *p = std::malloc(n)) return p;
    throw std::bad_alloc();
}
void operator delete(void *p) noexcept { std::free(p); }
void operator delete(void *p, size_t) noexcept { std::free(p); }

static void no_threads()
{
    hosthip::Stream s(0);
    nuctransfer::retain();
    warm(s);
    std::vector<double> h = values((size_t(5) << 20) + 3, 4), d(h.size()), r(h.size());
    refuse_new = true;
    const hipError_t up = nuctransfer::copy(d.data(), h.data(), 8 * h.size(), hipMemcpyHostToDevice, &s);
    const hipError_t down = nuctransfer::copy(r.data(), d.data(), 8 * d.size(), hipMemcpyDeviceToHost, &s);
    refuse_new = false;
    CHECK(up == hipSuccess && down == hipSuccess && r == h, "without memory for worker threads");
    nuctransfer::release();
}

int main(int argc, char **argv)
{
    const std::string what = argc > 1 ? argv[1] : "";
    if (what == "bytes") bytes();
    else if (what == "pinning") pinning();
    else if (what == "locks") locks();
    else if (what == "device") device();
    else if (what == "no_threads") no_threads();
    else { std::printf("unknown case\n"); return 2; }
    return failed != 0;
}

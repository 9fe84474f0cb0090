// The device memory that the library keeps between calls (mx_util.cpp), on a device that exists only here: the few HIP
// functions it calls are defined below and count bytes.  Run with the name of one check; exit status 0 means it holds.
#include <atomic>
#include <chrono>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <deque>
#include <map>
#include <mutex>
#include <new>
#include <string>
#include <thread>
#include <vector>

#include "mx_plan_parts.h"

namespace {

constexpr size_t GB = (size_t)1 << 30;

struct Device {
    std::mutex mu;
    size_t total = 256 * GB, used = 0, most = 0;
    std::map<void *, size_t> blocks;
    uintptr_t next = 0x10000;
    int frees = 0;
    std::atomic<int> streams{0};
    bool refuse = false;  // waits for the device
    hipError_t last = hipSuccess;
    // copies that run when they are waited for, in order; an event stands for those asked for before it
    struct Copy {
        void *to;
        const void *from;
        size_t n;
    };
    std::deque<Copy> copies;
    size_t done = 0;  // copies that have run
    std::map<hipEvent_t, size_t> events;
    size_t made = 0, plain = 0, pinned = 0;  // events; copies by hipMemcpy; bytes of pinned memory
    bool no_pinned = false;
    int copies_left = -1;  // so many are taken, the next is refused
    void run(size_t until)
    {
        for (; done < until; ++done) {
            std::memcpy(copies.front().to, copies.front().from, copies.front().n);
            copies.pop_front();
        }
    }
    size_t asked() const { return done + copies.size(); }
} device;

#define CHECK(x)                                                     \
    do {                                                             \
        if (!(x)) {                                                  \
            std::printf("line %d: %s does not hold\n", __LINE__, #x); \
            std::exit(1);                                            \
        }                                                            \
    } while (0)

void *take(size_t bytes)
{
    void *p = nullptr;
    CHECK(mx::dev_malloc(&p, bytes) == hipSuccess && p);
    return p;
}

}  // namespace

// (of the library only: the device's own bookkeeping does not count)
static thread_local long allocations_left = -1, own_business = 0;
void *operator new(size_t n)
{
    if (allocations_left >= 0 && own_business == 0 && allocations_left-- == 0) {
        allocations_left = 0;
        throw std::bad_alloc();
    }
    if (void *p = std::malloc(n)) return p;
    throw std::bad_alloc();
}
void operator delete(void *p) noexcept { std::free(p); }
void operator delete(void *p, size_t) noexcept { std::free(p); }
struct OwnBusiness {
    OwnBusiness() { ++own_business; }
    ~OwnBusiness() { --own_business; }
};

extern "C" {
hipError_t hipMalloc(void **p, size_t n)
{
    OwnBusiness own;
    std::lock_guard<std::mutex> hold(device.mu);
    if (device.used + n > device.total) return device.last = hipErrorOutOfMemory;
    *p = (void *)device.next;
    device.next += (n + 4095) / 4096 * 4096;
    device.blocks[*p] = n;
    device.used += n;
    device.most = std::max(device.most, device.used);
    return hipSuccess;
}
hipError_t hipFree(void *p)
{
    std::lock_guard<std::mutex> hold(device.mu);
    auto it = device.blocks.find(p);
    if (it == device.blocks.end()) std::abort();  // (freed twice)
    device.used -= it->second;
    device.blocks.erase(it);
    ++device.frees;
    return hipSuccess;
}
hipError_t hipGetDevice(int *d) { return *d = 0, hipSuccess; }
hipError_t hipMemGetInfo(size_t *f, size_t *t) { return *f = device.total - device.used, *t = device.total, hipSuccess; }
hipError_t hipDeviceSynchronize() { return device.refuse ? hipErrorStreamCaptureUnsupported : hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t)
{
    std::lock_guard<std::mutex> hold(device.mu);
    device.run(device.asked());
    return hipSuccess;
}
hipError_t hipMemcpyAsync(void *to, const void *from, size_t n, hipMemcpyKind, hipStream_t)
{
    std::lock_guard<std::mutex> hold(device.mu);
    if (device.copies_left >= 0 && device.copies_left-- == 0) return hipErrorInvalidValue;
    device.copies.push_back({to, from, n});
    return hipSuccess;
}
hipError_t hipMemcpy(void *to, const void *from, size_t n, hipMemcpyKind)
{
    {
        std::lock_guard<std::mutex> hold(device.mu);
        ++device.plain;
    }
    std::memcpy(to, from, n);
    return hipSuccess;
}
hipError_t hipHostMalloc(void **p, size_t n, unsigned)
{
    std::lock_guard<std::mutex> hold(device.mu);
    if (device.no_pinned) return device.last = hipErrorOutOfMemory;
    device.pinned += n;
    size_t *at = (size_t *)std::malloc(n + 64);
    *at = n;
    return *p = (char *)at + 64, hipSuccess;
}
hipError_t hipHostFree(void *p)
{
    std::lock_guard<std::mutex> hold(device.mu);
    CHECK(device.copies.empty());  // (nothing reads it any more)
    size_t *at = (size_t *)((char *)p - 64);
    device.pinned -= *at;
    std::free(at);
    return hipSuccess;
}
hipError_t hipEventCreateWithFlags(hipEvent_t *e, unsigned)
{
    std::lock_guard<std::mutex> hold(device.mu);
    *e = (hipEvent_t)(uintptr_t)(1000 + ++device.made);
    device.events[*e] = 0;
    return hipSuccess;
}
hipError_t hipEventRecord(hipEvent_t e, hipStream_t)
{
    std::lock_guard<std::mutex> hold(device.mu);
    device.events.at(e) = device.asked();
    return hipSuccess;
}
hipError_t hipEventSynchronize(hipEvent_t e)
{
    std::lock_guard<std::mutex> hold(device.mu);
    device.run(device.events.at(e));
    return hipSuccess;
}
hipError_t hipEventDestroy(hipEvent_t e)
{
    std::lock_guard<std::mutex> hold(device.mu);
    CHECK(device.events.erase(e) == 1);
    return hipSuccess;
}
hipError_t hipStreamCreate(hipStream_t *s)
{
    std::this_thread::sleep_for(std::chrono::milliseconds(2));
    *s = (hipStream_t)(uintptr_t)++device.streams;
    return hipSuccess;
}
hipError_t hipEventCreate(hipEvent_t *e) { return *e = (hipEvent_t)(uintptr_t)1, hipSuccess; }
const char *hipGetErrorString(hipError_t) { return ""; }
hipError_t hipGetLastError()
{
    const hipError_t e = device.last;
    device.last = hipSuccess;
    return e;
}
}

// Where the wait for the device is refused, no block becomes anybody's.
static void wait_refused()
{
    void *p = take(GB);
    device.refuse = true;
    {
        mx::IdleFrees idle;
        CHECK(mx::dev_free(p) == hipSuccess);
    }
    device.refuse = false;
    CHECK(device.frees == 1 && device.used == 0);
    CHECK(take(GB) != p);
}

// What lies idle is at most 1/128 of the device after every way of giving memory back.
static void bound()
{
    const size_t limit = device.total / 128;
    std::vector<void *> plan;
    for (int k = 0; k < 20; ++k) plan.push_back(take(GB));
    {
        mx::IdleFrees idle;  // a plan is destroyed
        for (void *p : plan) CHECK(mx::dev_free(p) == hipSuccess);
    }
    CHECK(device.used > 0 && device.used <= limit);
    for (int k = 1; k <= 40; ++k) {  // calls without a scope, each on a larger matrix
        void *p = take((size_t)k * 300 << 20);
        CHECK(mx::dev_free(p) == hipSuccess);
        CHECK(device.used <= limit);
    }
    for (int k = 0; k < 6; ++k) plan[k] = take(GB);
    {
        mx::MemScope scope(nullptr);
        for (int k = 0; k < 6; ++k) CHECK(mx::dev_free(plan[k]) == hipSuccess);
    }
    CHECK(device.used <= limit);
    mx::release_idle_memory();
    CHECK(device.used == 0);
}

// A block that nobody asks for is given back after 64 calls, also where those calls give nothing back themselves.
static void age()
{
    void *p = take(GB);
    CHECK(mx::dev_free(p) == hipSuccess);
    CHECK(device.used >= GB);
    for (int k = 0; k < 70; ++k) mx::MemScope scope(nullptr);
    CHECK(device.used == 0);
}

// A request that the device has room for once the scope's own blocks are given back is granted, and what a scope keeps for
// itself stays within its share.
static void scope_full()
{
    device.total = 10 * GB;
    {
        mx::MemScope scope(nullptr);
        std::vector<void *> part;
        for (int k = 0; k < 6; ++k) part.push_back(take(GB));
        for (void *p : part) CHECK(mx::dev_free(p) == hipSuccess);
        void *large = take(9 * GB);
        CHECK(mx::dev_free(large) == hipSuccess);
        void *none = nullptr;
        CHECK(mx::dev_malloc(&none, 11 * GB) == hipErrorOutOfMemory && !none);
        CHECK(hipGetLastError() == hipSuccess);
    }
    CHECK(device.used <= device.total / 128);
}
static void scope_share()
{
    const size_t share = device.total / 16;
    {
        mx::MemScope scope(nullptr);
        for (int k = 1; k <= 60; ++k) {
            void *p = take((size_t)k * 600 << 20);
            CHECK(mx::dev_free(p) == hipSuccess);
            CHECK(device.used <= share);
        }
    }
    CHECK(device.used <= device.total / 128);
}

// Threads that meet in the first call of a plan that needs a stream of its own get one and the same.
static void one_stream()
{
    for (int round = 0; round < 20; ++round) {
        mx_plan plan;
        device.streams = 0;
        std::vector<std::thread> threads;
        std::vector<hipStream_t> got(8, nullptr);
        for (int t = 0; t < 8; ++t)
            threads.emplace_back([&, t]() {
                if (!mxp::plan_stream(&plan)) got[t] = plan.stream;
            });
        for (auto &t : threads) t.join();
        CHECK(device.streams == 1 && plan.ev0 && plan.ev1);
        for (hipStream_t s : got) CHECK(s && s == plan.stream);
    }
}

// Host memory that runs out is an error of the allocation, or sends a block back to the device; nothing is thrown through
// the library's C entry points or out of a destructor, and nothing is lost.
static void host_memory()
{
    for (int after = 0; after < 12; ++after) {
        void *p = nullptr, *q = take(GB), *r = take(2 * GB);
        allocations_left = after;
        {
            mx::MemScope scope(nullptr);
            const hipError_t e = mx::dev_malloc(&p, 3 * GB);
            CHECK((e == hipSuccess) == (p != nullptr));
            CHECK(mx::dev_free(q) == hipSuccess);
            CHECK(mx::dev_free(p) == hipSuccess);
        }
        CHECK(mx::dev_free(r) == hipSuccess);
        allocations_left = -1;
        CHECK(device.used <= device.total / 128);
        mx::release_idle_memory();
        CHECK(device.used == 0 && device.blocks.empty());
    }
}

// Large copies go through pinned buffers, of which none is filled again before the device has read it (the copies here run as late as
// the waits allow); small ones, and all where there is no pinned memory, by hipMemcpy.
struct Bytes {
    std::vector<unsigned char> from, to;
    explicit Bytes(size_t n, unsigned seed) : from(n), to(n, 0)
    {
        for (auto &b : from) b = (unsigned char)((seed = seed * 1664525u + 1013904223u) >> 24);
    }
    hipError_t up() { return mx::copy_up(to.data(), from.data(), from.size()); }
    bool same() const { return from == to; }
};
static void copies()
{
    constexpr size_t MB = (size_t)1 << 20;
    for (const size_t n : {(size_t)0, (size_t)1, 8 * MB - 1}) {
        Bytes b(n, 3);
        const size_t plain = device.plain;
        CHECK(b.up() == hipSuccess && b.same() && device.plain == plain + 1 && device.pinned == 0);
    }
    for (const size_t n : {8 * MB, 8 * MB + 1, 12 * MB - 1, 16 * MB, 16 * MB + 1, 20 * MB, 33 * MB + 12345}) {
        Bytes b(n, (unsigned)n);
        const size_t plain = device.plain;
        CHECK(b.up() == hipSuccess && b.same() && device.plain == plain && device.events.empty());
        CHECK(device.pinned == 16 * MB && device.copies.empty());
    }
    mx_release_memory();
    CHECK(device.pinned == 0);
    Bytes b(9 * MB, 7);
    CHECK(b.up() == hipSuccess && b.same() && device.pinned == 16 * MB);
    mx_release_memory();
    device.no_pinned = true;
    Bytes c(9 * MB, 8);
    const size_t plain = device.plain;
    CHECK(c.up() == hipSuccess && c.same() && device.plain == plain + 1 && hipGetLastError() == hipSuccess);
}
static void copies_of_threads()
{
    std::vector<std::thread> threads;
    std::atomic<int> wrong{0};
    for (int t = 0; t < 4; ++t)
        threads.emplace_back([&, t]() {
            for (int k = 0; k < 6; ++k) {
                Bytes b(((size_t)10 << 20) + 4096 * t + k, 100 * t + k);
                if (b.up() != hipSuccess || !b.same()) ++wrong;
                if (t == 0) mx_release_memory();
            }
        });
    for (auto &t : threads) t.join();
    CHECK(wrong == 0 && device.events.empty() && device.copies.empty());
    mx_release_memory();
    CHECK(device.pinned == 0);
}
// A copy that the device refuses is an error; what was on its way is waited for.
static void copies_refused()
{
    for (int after = 0; after < 6; ++after) {
        Bytes b((size_t)40 << 20, 5);
        device.copies_left = after;
        CHECK(b.up() == hipErrorInvalidValue && device.copies.empty() && device.events.empty());
        device.copies_left = -1;
        CHECK(b.up() == hipSuccess && b.same());
    }
}

int main(int argc, char **argv)
{
    const std::map<std::string, void (*)()> checks = {{"copies", copies}, {"copies_of_threads", copies_of_threads}, {"copies_refused", copies_refused}, {"wait_refused", wait_refused}, {"bound", bound}, {"age", age}, {"scope_full", scope_full}, {"scope_share", scope_share}, {"one_stream", one_stream}, {"host_memory", host_memory}};
    const auto it = checks.find(argc > 1 ? argv[1] : "");
    if (it == checks.end()) return 2;
    it->second();
    return 0;
}

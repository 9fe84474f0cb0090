// Error text, binary16 conversions and the device memory kept between calls, shared by the host code.
#include <algorithm>
#include <cstdlib>
#include <cstring>
#include <iterator>
#include <map>
#include <mutex>
#include <new>
#include <unordered_map>

#include "mx_device.h"
#include "mx_internal.h"

namespace mx {

static thread_local std::string g_error;

void set_error(const std::string &msg) { g_error = msg; }

// One set for the process (the planners read it from OpenMP workers too).  It is rewritten only when the
// environment reads differently from the last time, so threads that make plans side by side under one
// environment never write it.
static Options g_options;
static std::mutex g_options_mu;
const Options &opt() { return g_options; }
static bool same(const Options &a, const Options &b)
{
    return a.tile_gate == b.tile_gate && a.csr_dict == b.csr_dict && a.no_strips == b.no_strips && a.no_blocks == b.no_blocks &&
           a.strips_apart == b.strips_apart && a.csr_kernel == b.csr_kernel && a.csr_fused == b.csr_fused && a.csr_keep == b.csr_keep && a.autotune == b.autotune &&
           a.layout_host == b.layout_host && a.slice_cap == b.slice_cap && a.split_len == b.split_len && a.csr_npt == b.csr_npt &&
           a.tile_per == b.tile_per && a.csr_reduce == b.csr_reduce && a.csr_col16 == b.csr_col16 && a.plan_log == b.plan_log;
}
void refresh_options()
{
    Options o;
    auto text = [](const char *name) { return std::getenv(name); };
    auto number = [&](const char *name, int unset) {
        const char *e = text(name);
        return e ? std::atoi(e) : unset;
    };
    if (const char *e = text("MX_TILE_GATE")) {
        const double v = std::atof(e);
        if (v >= 0.0 && v <= 1.0) o.tile_gate = v;
    }
    o.csr_dict = number("MX_CSR_DICT", 1);
    o.no_strips = number("MX_NO_STRIPS", 0) != 0;
    o.no_blocks = number("MX_NO_BLOCKS", 0) != 0;
    o.strips_apart = number("MX_STRIPS_APART", 0) != 0;
    if (const char *e = text("MX_CSR_KERNEL")) o.csr_kernel = !std::strcmp(e, "rows") ? 1 : !std::strcmp(e, "slices") ? 2 : !std::strcmp(e, "split") ? 3 : 0;
    if (const char *e = text("MX_CSR_FUSED")) o.csr_fused = std::atoi(e) ? 1 : 0;
    if (const char *e = text("MX_CSR_KEEP")) o.csr_keep = std::atoi(e) ? 1 : 0;
    o.autotune = number("MX_PLAN_AUTOTUNE", 0) != 0;
    if (const char *e = text("MX_LAYOUT")) o.layout_host = !std::strcmp(e, "host");
    o.slice_cap = number("MX_SLICE_CAP", 0);
    o.split_len = number("MX_SPLIT_LEN", 0);
    o.csr_npt = number("MX_CSR_NPT", 0);
    o.tile_per = number("MX_TILE_PER", 0);
    if (const char *e = text("MX_CSR_REDUCE")) o.csr_reduce = !std::strcmp(e, "rows") ? 1 : !std::strcmp(e, "scan") ? 2 : 0;
    o.csr_col16 = number("MX_CSR_COL16", 1) != 0;
    o.plan_log = number("MX_PLAN_LOG", 0) != 0;
    std::lock_guard<std::mutex> lock(g_options_mu);
    if (!same(g_options, o)) g_options = o;
}

uint16_t f64_to_f16_bits(double v)
{
    uint64_t b;
    std::memcpy(&b, &v, 8);
    const uint16_t sign = (uint16_t)((b >> 48) & 0x8000u);
    const uint64_t ab = b & 0x7fffffffffffffffull;
    if (ab >= 0x7ff0000000000000ull) return (uint16_t)(sign | (ab == 0x7ff0000000000000ull ? 0x7c00u : 0x7e00u));
    const int e = (int)(ab >> 52) - 1023;
    uint64_t m = ab & 0xfffffffffffffull;
    if (e > 15) return (uint16_t)(sign | 0x7c00u);
    if (e >= -14) {
        uint32_t h = ((uint32_t)(e + 15) << 10) | (uint32_t)(m >> 42);
        const uint64_t rem = m & ((1ull << 42) - 1), half = 1ull << 41;
        if (rem > half || (rem == half && (h & 1u))) ++h;  // a carry into the exponent is the right answer
        return (uint16_t)(sign | h);
    }
    if (e < -25) return sign;
    m |= 1ull << 52;
    const int shift = 42 + (-14 - e);  // 43..53
    uint32_t hm = (uint32_t)(m >> shift);
    const uint64_t rem = m & ((1ull << shift) - 1), half = 1ull << (shift - 1);
    if (rem > half || (rem == half && (hm & 1u))) ++hm;
    return (uint16_t)(sign | hm);
}

float f16_bits_to_f32(uint16_t h)
{
    const uint32_t sign = (uint32_t)(h & 0x8000u) << 16;
    const uint32_t ex = (h >> 10) & 0x1fu;
    const uint32_t man = h & 0x3ffu;
    float out;
    if (ex == 0) {
        // subnormal or zero: man * 2^-24, exact in binary32
        out = (float)man * (1.0f / 16777216.0f);
        uint32_t bits;
        std::memcpy(&bits, &out, 4);
        bits |= sign;
        std::memcpy(&out, &bits, 4);
        return out;
    }
    uint32_t bits = ex == 31 ? (sign | 0x7f800000u | (man << 13)) : (sign | ((ex + 112u) << 23) | (man << 13));
    std::memcpy(&out, &bits, 4);
    return out;
}

}  // namespace mx

extern "C" const char *mx_last_error(void) { return mx::g_error.c_str(); }

extern "C" uint16_t mx_f32_to_f16(float f) { return mx::f64_to_f16_bits((double)f); }
extern "C" float mx_f16_to_f32(uint16_t h) { return mx::f16_bits_to_f32(h); }

// ---- device memory kept from one call to the next --------------------------------------------------------
namespace mx {
namespace {

// A block of at least this many bytes is handed out for a request when it is not more than an eighth (and
// 64 KB) larger.
size_t block_bytes(size_t n)
{
    if (n < 512) return 512;
    size_t step = 256;  // an eighth of the largest power of two in n, at least 256 bytes, at most 2 MB
    while (step * 16 <= n && step < ((size_t)2 << 20)) step *= 2;
    return (n + step - 1) / step * step;
}

struct Block {
    size_t bytes;
    int dev;
};
struct Idle {
    void *p;
    uint64_t stamp;  // number of the call that gave it back
};
constexpr int kPoolDevices = 64;
constexpr uint64_t kPoolCalls = 64;   // a block nobody has asked for in so many calls goes back to the device
constexpr size_t kPoolShare = 128;    // idle blocks hold at most this fraction of a device's memory (2.25 GB of 288)
constexpr size_t kScopeShare = 16;    // what a thread has given back inside its scope, at most (18 GB)

struct Pool {
    std::mutex mu;
    std::unordered_map<void *, Block> blocks;            // every block made here, in use or idle
    std::multimap<size_t, Idle> idle[kPoolDevices];      // by size; no work on the device touches them any more
    size_t idleBytes[kPoolDevices] = {}, limit[kPoolDevices] = {};
    uint64_t calls = 0;
};
Pool &pool()
{
    static Pool *p = new Pool();  // (never destroyed: plans may be released by destructors that run after this file's)
    return *p;
}

// What the calling thread has given back inside its current MemScope.
struct ThreadScope {
    int depth = 0, idleFrees = 0;
    bool waited = false;  // the last IdleFrees' wait for the device was granted and ended
    hipStream_t stream = nullptr;
    std::multimap<size_t, void *> freed;
    size_t freedBytes = 0;
};
thread_local ThreadScope t_scope;

// Blocks beyond the bound, and blocks nobody has asked for in a while (`all`: every block), go back to the device, oldest first,
// of equally old ones the largest: a call that passes the bound gives back a few large blocks, not dozens of small ones (plan
// and first product of 45 million binary16 entries 27.0 -> 15.8 ms)
void trim(Pool &P, bool all)
{
    for (int dev = 0; dev < kPoolDevices; ++dev)
        for (;;) {
            void *p;
            {
                std::lock_guard<std::mutex> hold(P.mu);
                auto &I = P.idle[dev];
                auto oldest = I.end();
                for (auto it = I.begin(); it != I.end(); ++it)
                    if (oldest == I.end() || it->second.stamp <= oldest->second.stamp) oldest = it;
                if (oldest == I.end() || !(all || P.idleBytes[dev] > P.limit[dev] || oldest->second.stamp + kPoolCalls < P.calls)) break;
                P.idleBytes[dev] -= oldest->first;
                p = oldest->second.p;
                P.blocks.erase(p);
                I.erase(oldest);
            }
            (void)hipFree(p);
        }
}
// (with the lock held) false where host memory has run out: the block goes back to the device then
bool put_idle(Pool &P, void *p, const Block &b)
{
    try {
        P.idle[b.dev].emplace(b.bytes, Idle{p, P.calls});
    } catch (const std::bad_alloc &) {
        return false;
    }
    P.idleBytes[b.dev] += b.bytes;
    return true;
}
// What the thread has given back inside its scope goes back to the device, the largest block first, until at most `keep` bytes
// are left -- after a wait for the scope's stream; nothing does where that fails.
void shrink_scope(Pool &P, ThreadScope &T, size_t keep)
{
    if (T.freedBytes <= keep || hipStreamSynchronize(T.stream) != hipSuccess) return;
    while (T.freedBytes > keep) {
        const auto it = std::prev(T.freed.end());
        void *p = it->second;
        T.freedBytes -= it->first;
        T.freed.erase(it);
        {
            std::lock_guard<std::mutex> hold(P.mu);
            P.blocks.erase(p);
        }
        (void)hipFree(p);
    }
}
bool fits(size_t have, size_t need) { return have <= need + need / 8 + 65536; }

}  // namespace

hipError_t dev_malloc(void **out, size_t bytes)
{
    *out = nullptr;
    int dev = 0;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess) return e;
    if (dev < 0 || dev >= kPoolDevices) return hipMalloc(out, bytes);
    const size_t need = block_bytes(bytes);
    Pool &P = pool();
    ThreadScope &T = t_scope;
    if (T.depth > 0) {
        auto it = T.freed.lower_bound(need);
        if (it != T.freed.end() && fits(it->first, need)) {
            *out = it->second;
            T.freedBytes -= it->first;
            T.freed.erase(it);
            return hipSuccess;
        }
    }
    {
        std::lock_guard<std::mutex> hold(P.mu);
        auto it = P.idle[dev].lower_bound(need);
        if (it != P.idle[dev].end() && fits(it->first, need)) {
            *out = it->second.p;
            P.idleBytes[dev] -= it->first;
            P.idle[dev].erase(it);
            return hipSuccess;
        }
    }
    void *p = nullptr;
    e = hipMalloc(&p, need);
    if (e == hipErrorOutOfMemory) {  // what lies idle here, or waits in this scope, may be what is missing
        (void)hipGetLastError();
        shrink_scope(P, T, 0);
        release_idle_memory();
        e = hipMalloc(&p, need);
    }
    if (e != hipSuccess) {
        (void)hipGetLastError();  // (a caller that goes on without the memory must not meet the error at its next launch)
        return e;
    }
    std::unique_lock<std::mutex> hold(P.mu);
    if (P.limit[dev] == 0) {
        size_t freeB = 0, total = 0;
        if (hipMemGetInfo(&freeB, &total) != hipSuccess) {
            (void)hipGetLastError();
            total = (size_t)16 << 30;
        }
        P.limit[dev] = std::max<size_t>(total / kPoolShare, 1);
    }
    try {
        P.blocks[p] = Block{need, dev};
    } catch (const std::bad_alloc &) {
        hold.unlock();
        (void)hipFree(p);
        return hipErrorOutOfMemory;
    }
    *out = p;
    return hipSuccess;
}

hipError_t dev_free(void *p)
{
    if (!p) return hipSuccess;
    Pool &P = pool();
    ThreadScope &T = t_scope;
    if (T.depth == 0 && T.idleFrees == 0) {
        IdleFrees one;
        return dev_free(p);
    }
    Block b{};
    size_t scopeLimit = 0;
    {
        std::lock_guard<std::mutex> hold(P.mu);
        auto it = P.blocks.find(p);
        int dev = -1;
        if (it == P.blocks.end() || hipGetDevice(&dev) != hipSuccess || dev != it->second.dev || (T.idleFrees > 0 && !T.waited)) {
            // not made here, on another device than the current one, or still read by work that could not be waited for (a plan
            // dropped while a stream is captured): the plain way
            if (it != P.blocks.end()) P.blocks.erase(it);
            b.bytes = 0;
        } else {
            b = it->second;
            scopeLimit = P.limit[b.dev] * (kPoolShare / kScopeShare);
            bool kept = true;
            if (T.idleFrees > 0) {
                if (put_idle(P, p, b)) return hipSuccess;
                kept = false;
            } else {
                try {
                    T.freed.emplace(b.bytes, p);
                } catch (const std::bad_alloc &) {
                    kept = false;
                }
            }
            if (!kept) {
                P.blocks.erase(it);
                b.bytes = 0;
            }
        }
    }
    if (b.bytes == 0) return hipFree(p);
    T.freedBytes += b.bytes;
    shrink_scope(P, T, scopeLimit);
    return hipSuccess;
}

void release_idle_memory() { trim(pool(), true); }

MemScope::MemScope(hipStream_t s)
{
    ThreadScope &T = t_scope;
    // (a call inside another one works on the same stream -- every caller here hands its own on -- or is done with
    // the memory it gave back when it returns)
    if (T.depth++ == 0) T.stream = s;
}
MemScope::~MemScope()
{
    ThreadScope &T = t_scope;
    if (--T.depth > 0) return;
    const bool idle = T.freed.empty() || hipStreamSynchronize(T.stream) == hipSuccess;
    Pool &P = pool();
    {
        std::lock_guard<std::mutex> hold(P.mu);
        ++P.calls;
    }
    for (auto &f : T.freed) {
        {
            std::lock_guard<std::mutex> hold(P.mu);
            auto it = P.blocks.find(f.second);
            if (it != P.blocks.end()) {
                if (idle && put_idle(P, f.second, it->second)) continue;
                P.blocks.erase(it);
            }
        }
        (void)hipFree(f.second);
    }
    T.freed.clear();
    T.freedBytes = 0;
    trim(P, false);
}

IdleFrees::IdleFrees()
{
    t_scope.waited = hipDeviceSynchronize() == hipSuccess;
    ++t_scope.idleFrees;
}
IdleFrees::~IdleFrees()
{
    if (--t_scope.idleFrees > 0) return;
    Pool &P = pool();
    {
        std::lock_guard<std::mutex> hold(P.mu);
        ++P.calls;
    }
    trim(P, false);
}

}  // namespace mx

extern "C" void mx_release_memory(void)
{
    mx::release_staging();
    mx::release_idle_memory();
}

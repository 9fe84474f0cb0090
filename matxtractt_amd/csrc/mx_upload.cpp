// Large copies from memory that a caller allocated as it liked.
#include <algorithm>
#include <cstring>
#include <mutex>

#include "mx_device.h"

namespace {
struct Staging {
    std::mutex lock;
    unsigned char *pinned = nullptr;
};
constexpr size_t kStage = (size_t)4 << 20;
constexpr int kStages = 4;
Staging &staging()
{
    static Staging *s = new Staging();  // (not destroyed: the runtime may be gone by then)
    return *s;
}
}  // namespace

void mx::release_staging()
{
    Staging &S = staging();
    std::lock_guard<std::mutex> hold(S.lock);
    if (S.pinned) (void)hipHostFree(S.pinned);
    S.pinned = nullptr;
}

hipError_t mx::copy_up(void *dst, const void *src, size_t bytes)
{
    Staging &S = staging();
    std::unique_lock<std::mutex> hold(S.lock, std::defer_lock);
    if (bytes < 2 * kStage || !hold.try_lock()) return hipMemcpy(dst, src, bytes, hipMemcpyHostToDevice);
    if (!S.pinned && hipHostMalloc((void **)&S.pinned, kStage * kStages, hipHostMallocPortable) != hipSuccess) {
        (void)hipGetLastError();
        S.pinned = nullptr;
        return hipMemcpy(dst, src, bytes, hipMemcpyHostToDevice);
    }
    hipEvent_t read[kStages] = {};
    hipError_t e = hipSuccess;
    int made = 0;
    while (made < kStages && e == hipSuccess) e = hipEventCreateWithFlags(&read[made], hipEventDisableTiming), made += e == hipSuccess;
    size_t at = 0;
    for (int i = 0; at < bytes && e == hipSuccess; ++i) {
        const int b = i % kStages;
        const size_t n = std::min(kStage, bytes - at);
        if (i >= kStages) e = hipEventSynchronize(read[b]);  // the device is done with what the buffer held
        if (e != hipSuccess) break;
        unsigned char *to = S.pinned + (size_t)b * kStage;
        const unsigned char *from = (const unsigned char *)src + at;
        constexpr size_t piece = (size_t)256 << 10;
        const int pieces = (int)((n + piece - 1) / piece);
// (by as many threads as the host's other loops: a team of another size ends threads and starts them again, 0.15 ms of a plan that both are in)
#pragma omp parallel for schedule(static)
        for (int k = 0; k < pieces; ++k) std::memcpy(to + k * piece, from + k * piece, std::min(piece, n - k * piece));
        e = hipMemcpyAsync((unsigned char *)dst + at, to, n, hipMemcpyHostToDevice, nullptr);
        if (e == hipSuccess) e = hipEventRecord(read[b], nullptr);
        at += n;
    }
    const hipError_t waited = hipStreamSynchronize(nullptr);
    for (int b = 0; b < made; ++b) (void)hipEventDestroy(read[b]);
    return e != hipSuccess ? e : waited;
}

// The part of the slice layout that looks at chunks only, on the device (mx_chunks.hip), for mx_layout.hip.
#pragma once
#include <hip/hip_runtime.h>

#include <string>

#include "mx_device.h"
#include "mx_internal.h"

namespace mxl {

constexpr int kBlock = 256;
inline dim3 grid(long long n) { return dim3((unsigned)(((n > 1 ? n : 1) + kBlock - 1) / kBlock)); }

struct Buf {  // device memory released at scope exit unless taken
    void *p = nullptr;
    Buf() = default;
    Buf(const Buf &) = delete;
    Buf &operator=(const Buf &) = delete;
    ~Buf() { release(); }
    void release()
    {
        if (p) (void)mx::dev_free(p);
        p = nullptr;
    }
    template <typename T>
    T *as() const
    {
        return (T *)p;
    }
    void *take()
    {
        void *q = p;
        p = nullptr;
        return q;
    }
};

// What plan_slice_chunks decides (SlicePlan), in device memory: the descriptors that the kernels read and, for every
// chunk in its final numbering, where it comes from and at which step of the streams it starts.
struct ChunkPlan {
    int nWG = 0, maxWgChunks = 0;
    long long totalSteps = 0, totalChunks = 0;
    Buf wgDesc, waveDesc, chunkEnd;
    const int *chunkFirst = nullptr, *chunkN = nullptr, *chunkSteps = nullptr;  // (in `made`)
    const long long *chunkStep0 = nullptr;
    Buf made;
};
// Chunks of 64 virtual rows per slice from their order by (slice, length descending): virtual row `sorted[i]` has vLen[sorted[i]] entries
// and slice q holds the places whose keys lie in [q * perSlice, (q + 1) * perSlice).  One wait.
int plan_chunks_device(mx_dtype dtype, int budget, int S, int nV, const unsigned *sortedKey, unsigned perSlice, const int *sorted,
                       const int *vLen, ChunkPlan &P, hipStream_t s);

// The one-launch form's part of a plan.
struct FusedPlan {
    int nGroups = 0, maxWgGroups = 0, places = 0;
    Buf wgGroups, groupNeed;
};
// Whether plan_fused_device makes the plan: (XCD, slice) and a length are one digit each, and there are enough virtual rows (14 thousand: the plan
// of a power law of 12000 rows 467 us on the device, 427 on the host; 118 thousand: 940 and 1230).
bool fused_plan_on_device(int S, int cap, int nV);
// plan_fused_records on the device: *taken, with `sorted` (the order in which the virtual rows are laid out), P and F filled, when the form is taken;
// otherwise nothing is to be used.  vRow, vSlice, vLen: the virtual rows in the order of the rows.  One wait.
int plan_fused_device(mx_dtype dtype, int budget, int S, int rows, int nnz, int cap, int nV, int mode, const int *rowPtr, const int *segPtr,
                      const int *vRow, const int *vSlice, const int *vLen, int *sorted, ChunkPlan &P, FusedPlan &F, bool *taken, hipStream_t s);
// fused_targets on the device: target [totalChunks * 64 + 64]
int fused_targets_device(int nGroups, int places, long long totalChunks, const int *segPtr, const int *segIdx, const int *vRow, int nV, int *target,
                         hipStream_t s);

}  // namespace mxl

#define MXL_TRY(call)                                                                                 \
    do {                                                                                              \
        hipError_t e_ = (call);                                                                       \
        if (e_ != hipSuccess) {                                                                       \
            mx::set_error(std::string("slice layout on the device: ") + #call + ": " + hipGetErrorString(e_)); \
            return e_ == hipErrorOutOfMemory ? MX_ERR_ALLOC : MX_ERR_DEVICE;                          \
        }                                                                                             \
    } while (0)

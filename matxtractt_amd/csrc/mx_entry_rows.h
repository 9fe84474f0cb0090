// Device code shared by the kernels that make plans (mx_prep.hip, mx_layout.hip, mx_hybrid.hip): which row an
// entry of a CSR matrix belongs to, for a tile of consecutive entries at a time.
#pragma once
#include <hip/hip_runtime.h>

#include <algorithm>

#include "mx_device.h"

namespace mxr {

constexpr int kBlock = 256;
constexpr int kPer = 4;                  // entries per thread
constexpr int kTile = kBlock * kPer;     // entries per workgroup
inline dim3 tile_grid(long long n) { return dim3((unsigned)((std::max<long long>(n, 1) + kTile - 1) / kTile)); }

template <int THREADS, int PER>
struct TileRowsOf {
    int row[THREADS * PER];
    int top[THREADS / 64];
};
using TileRows = TileRowsOf<kBlock, kPer>;

// The rows of the entries [t0, t0 + THREADS * PER) of a matrix with n entries, by a workgroup of THREADS threads:
// T.row[i] is the row of entry t0 + i (the last r < rows with ptr[r] <= t0 + i).  A search of the row pointers per entry is
// twenty dependent loads of its own for a matrix of a million rows, and the kernels that did so spent most of
// their time on them; here a workgroup searches once, 64 pointers at a look, marks where the rows behind begin, and
// a running maximum does the rest.  Whatever stands in ptr, the rows found lie in [0, rows) and no access outside ptr[0 .. rows]
// is made (rows >= 1; entry points whose arrays are not looked at beforehand rely on that).  Every thread of the workgroup has to come here.
template <int THREADS, int PER>
__device__ __forceinline__ void tile_rows(const int *__restrict__ ptr, int rows, int n, int t0, TileRowsOf<THREADS, PER> &T)
{
    constexpr int kBlock = THREADS, kPer = PER, kTile = THREADS * PER;
    const int tid = threadIdx.x, lane = tid & 63;
    int lo = 0, hi = rows;  // the row of entry t0 lies in [lo, hi)
    while (hi - lo > 1) {
        const int step = (hi - lo + 63) / 64;
        const long long i = lo + (long long)lane * step;
        const unsigned long long not_above = __ballot(i < hi && (lane == 0 || ptr[i < hi ? i : lo] <= t0));
        lo += (63 - __builtin_clzll(not_above)) * step;
        hi = min(hi, lo + step);
    }
#pragma unroll
    for (int k = 0; k < kPer; ++k) T.row[k * kBlock + tid] = 0;
    __syncthreads();
    const int size = min(n - t0, kTile);
    // Where nearly all rows are without entries, walking them takes longer than a search per entry: the row
    // 8 * kTile further on begins inside the tile.
    if (rows - lo > 8 * kTile && (long long)ptr[lo + 8 * kTile] < (long long)t0 + size) {
        for (int i = tid; i < size; i += kBlock) {
            int a = lo, b = rows - 1;
            while (a < b) {
                const int mid = a + (b - a + 1) / 2;
                if ((long long)ptr[mid] - t0 <= i) a = mid;
                else b = mid - 1;
            }
            T.row[i] = a;
        }
        __syncthreads();
        return;
    }
    for (int r = mx::next_of(lo, rows, 1 + tid); r < rows; r = mx::next_of(r, rows, kBlock)) {
        const long long at = (long long)ptr[r] - t0;
        if (at >= size) break;
        if (at >= 0 && ptr[r + 1] > ptr[r]) T.row[at] = r - lo;
    }
    __syncthreads();
    int m[kPer];
#pragma unroll
    for (int k = 0; k < kPer; ++k) {
        m[k] = T.row[tid * kPer + k];
        if (k) m[k] = max(m[k], m[k - 1]);
    }
    int before = m[kPer - 1];  // running maximum over the threads
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
        const int o = __shfl_up(before, off);
        if (lane >= off) before = max(before, o);
    }
    if (lane == 63) T.top[tid >> 6] = before;
    before = __shfl_up(before, 1);
    if (lane == 0) before = 0;
    __syncthreads();
    for (int w = 0; w < (tid >> 6); ++w) before = max(before, T.top[w]);
#pragma unroll
    for (int k = 0; k < kPer; ++k) T.row[tid * kPer + k] = lo + max(before, m[k]);
    __syncthreads();
}

}  // namespace mxr

// Entries put in order inside their rows, shared by the kernels that make plans (mx_prep.hip, mx_layout.hip).
//
// A row's entries already lie together, so nothing has to be sorted across rows: a row is put in order inside one
// workgroup, in registers and LDS, and the matrix is read once and written once.  (A radix sort of all entries by
// {row, key} moves 24 bytes an entry through memory for every eight bits of the two together, six times for a million
// rows and columns: 0.83 ms for 15.8 million entries, and 28 bytes an entry of working memory; this takes 0.31 to 0.44 ms and none.  Without that
// memory the plan of such a matrix stays inside what is kept from one call to the next: 15.4 -> 7.2 ms, 5.7 of them hipFree.)
//
//   rows of at most kShort entries   several to a workgroup, 1536 entries and the rest of the last row at a time
//   rows of at most 2048/4096/8192   one to a workgroup of 256/512/1024 threads, from lists made on the device
//   longer rows                      not here: the caller looks at the count of them and takes the radix sort
//
// The order inside a row is by key, equal keys as they were: the place an entry had is part of what is compared, so no two
// are equal and any sorting network gives the one result.  The network is bitonic: it needs no counts, its first
// three distances stay inside a thread's eight entries, the next six are lane exchanges, and only the largest go through LDS.
#pragma once
#include <hip/hip_runtime.h>

#include <algorithm>

namespace mxs {

constexpr int kThreads = 256, kPer = 8;       // of a workgroup of short rows
constexpr int kRoom = kThreads * kPer;        // entries it has room for
constexpr int kShort = 512;                   // entries of a short row at most
constexpr int kTile = kRoom - kShort;         // rows that begin in so many entries belong to one workgroup
constexpr int kClasses = 3;                   // of longer rows: 2048, 4096 and 8192 entries at most
constexpr int kLongest = 8192;
constexpr int kPad = 8;                       // LDS: consecutive entries of a thread lie kThreads + kPad apart

// What the host reads back: rows of each class, and of none.
struct RowClasses {
    int n[kClasses + 1];
};
// ints of the lists of one matrix: rows of more than 512, 2048 and 4096 entries are at most so many
inline size_t list_ints(long long entries) { return (size_t)(entries / kShort + entries / 2048 + entries / 4096 + 3); }

// count[c] rows of class c, in list + list_at(c, entries)
static __global__ __launch_bounds__(256) void row_classes_kernel(const int *__restrict__ ptr, int rows, int entries, int *__restrict__ list,
                                                                 int *__restrict__ count)
{
    __shared__ int here[kClasses + 1], first[kClasses + 1];  // (one atomic per workgroup and class)
    const int tid = threadIdx.x, r = blockIdx.x * 256 + tid;
    if (tid <= kClasses) here[tid] = 0;
    __syncthreads();
    const int n = r < rows ? ptr[r + 1] - ptr[r] : 0;
    const int c = n <= kShort ? -1 : n <= 2048 ? 0 : n <= 4096 ? 1 : n <= kLongest ? 2 : 3;
    const int at = c < 0 ? 0 : atomicAdd(&here[c], 1);
    __syncthreads();
    if (tid <= kClasses && here[tid]) first[tid] = atomicAdd(&count[tid], here[tid]);
    __syncthreads();
    // (the bound holds for pointers that nobody has looked at yet, too)
    const int base[kClasses + 1] = {0, entries / kShort + 1, entries / kShort + entries / 2048 + 2, entries / kShort + entries / 2048 + entries / 4096 + 3};
    if (c >= 0 && c < kClasses && first[c] + at < base[c + 1] - base[c]) list[base[c] + first[c] + at] = r;
}
inline size_t list_at(int c, long long entries)
{
    return c == 0 ? 0 : c == 1 ? (size_t)(entries / kShort + 1) : (size_t)(entries / kShort + entries / 2048 + 2);
}

__device__ __forceinline__ void order_pair(unsigned long long &a, unsigned long long &b, bool up)
{
    const unsigned long long x = a, y = b;
    const bool swap = (y < x) == up;
    a = swap ? y : x;
    b = swap ? x : y;
}

// The THREADS * kPer values of a workgroup in ascending order; thread t ends with the places kPer * t and on.
template <int THREADS>
__device__ __forceinline__ void sort_workgroup(unsigned long long (&v)[kPer], unsigned long long *__restrict__ lds)
{
    const int tid = threadIdx.x;
    auto within = [&](bool up) {
#pragma unroll
        for (int d = 4; d; d >>= 1)
#pragma unroll
            for (int j = 0; j < kPer; ++j)
                if (!(j & d)) order_pair(v[j], v[j | d], up);
    };
#pragma unroll
    for (int j = 0; j < kPer; j += 2) order_pair(v[j], v[j + 1], !(j & 2));
#pragma unroll
    for (int d = 2; d; d >>= 1)
#pragma unroll
        for (int j = 0; j < kPer; ++j)
            if (!(j & d)) order_pair(v[j], v[j | d], !(j & 4));
    within(!(tid & 1));
    for (int k = 2; k <= THREADS; k <<= 1) {  // (in threads: runs of kPer * k places)
        const bool up = (tid & k) == 0;
        int m = k >> 1;
        for (; m >= 64; m >>= 1) {
            const bool low = ((tid & m) == 0) == up;
#pragma unroll
            for (int j = 0; j < kPer; ++j) lds[j * (THREADS + kPad) + tid] = v[j];
            __syncthreads();
#pragma unroll
            for (int j = 0; j < kPer; ++j) {
                const unsigned long long o = lds[j * (THREADS + kPad) + (tid ^ m)];
                v[j] = (o < v[j]) == low ? o : v[j];
            }
            __syncthreads();
        }
        for (; m; m >>= 1) {
            const bool low = ((tid & m) == 0) == up;
#pragma unroll
            for (int j = 0; j < kPer; ++j) {
                const unsigned long long o = __shfl_xor(v[j], m);
                v[j] = (o < v[j]) == low ? o : v[j];
            }
        }
        within(up);
    }
#pragma unroll
    for (int j = 0; j < kPer; ++j) lds[j * (THREADS + kPad) + tid] = v[j];
    __syncthreads();
}
template <int THREADS>
__device__ __forceinline__ unsigned long long sorted_at(const unsigned long long *__restrict__ lds, int place)
{
    return lds[(place & (kPer - 1)) * (THREADS + kPad) + place / kPer];
}

// The first row r of [0, rows] with ptr[r] >= at (rows, where there is none), by one wave, 64 pointers at a look.
__device__ __forceinline__ int first_row_from(const int *__restrict__ ptr, int rows, long long at)
{
    const int lane = threadIdx.x & 63;
    int lo = 0, hi = rows;
    while (lo < hi) {
        const int step = (hi - lo + 63) / 64;
        const long long i = lo + (long long)lane * step;
        const int below = __popcll(__ballot(i < hi && ptr[i < hi ? i : lo] < at));
        if (below == 0) break;
        hi = (int)min((long long)hi, lo + (long long)below * step);
        lo += (below - 1) * step + 1;
    }
    return lo;
}

// IO: unsigned key(row, entry); void put(row, place in the row, key, entry, place in the matrix).
// ptr ascends from 0 to `entries`; an entry's key is asked for once, and every entry of a row of at most kShort is put once.
template <typename IO>
__global__ __launch_bounds__(kThreads) void sort_short_rows_kernel(const int *__restrict__ ptr, int rows, IO io)
{
    __shared__ unsigned long long lds[kPer * (kThreads + kPad)];
    __shared__ int rowOf[kRoom];
    __shared__ int top[kThreads / 64];
    const int tid = threadIdx.x, lane = tid & 63;
    const int r0 = first_row_from(ptr, rows, (long long)blockIdx.x * kTile);
    const int r1 = first_row_from(ptr, rows, (long long)(blockIdx.x + 1) * kTile);
    if (r0 >= r1) return;
    const int p0 = ptr[r0], size = min(ptr[r1] - p0, kRoom);
    if (size <= 0) return;
    // ---- the row of every entry
    if (r1 - r0 <= 8 * kRoom) {
#pragma unroll
        for (int j = 0; j < kPer; ++j) rowOf[j * kThreads + tid] = 0;
        __syncthreads();
        for (int r = r0 + tid; r < r1; r += kThreads) {
            const int at = ptr[r] - p0;
            if (at < size && ptr[r + 1] - p0 > at) rowOf[at] = r - r0;
        }
        __syncthreads();
        int m[kPer];
#pragma unroll
        for (int j = 0; j < kPer; ++j) {
            m[j] = rowOf[tid * kPer + j];
            if (j) m[j] = max(m[j], m[j - 1]);
        }
        int before = m[kPer - 1];
#pragma unroll
        for (int off = 1; off < 64; off <<= 1) {
            const int o = __shfl_up(before, off);
            if (lane >= off) before = max(before, o);
        }
        if (lane == 63) top[tid >> 6] = before;
        before = __shfl_up(before, 1);
        if (lane == 0) before = 0;
        __syncthreads();
        for (int w = 0; w < (tid >> 6); ++w) before = max(before, top[w]);
#pragma unroll
        for (int j = 0; j < kPer; ++j) rowOf[tid * kPer + j] = max(before, m[j]);
    } else {  // mostly rows without entries: walking all of them would take longer than a search per entry
        for (int i = tid; i < kRoom; i += kThreads) {
            int lo = r0, hi = r1 - 1;
            while (lo < hi) {
                const int mid = lo + (hi - lo + 1) / 2;
                if (ptr[mid] - p0 <= i) lo = mid;
                else hi = mid - 1;
            }
            rowOf[i] = lo - r0;
        }
    }
    __syncthreads();
    // ---- sorted by {where the row begins, key, place}
    unsigned long long v[kPer];
#pragma unroll
    for (int j = 0; j < kPer; ++j) {
        const int i = j * kThreads + tid;
        v[j] = ~0ull;
        if (i < size) {
            const int r = r0 + rowOf[i];
            v[j] = ((unsigned long long)(unsigned)(ptr[r] - p0) << 44) | ((unsigned long long)io.key(r, p0 + i) << 12) | (unsigned)i;
        }
    }
    sort_workgroup<kThreads>(v, lds);
#pragma unroll
    for (int j = 0; j < kPer; ++j) {
        const int i = j * kThreads + tid;
        if (i >= size) continue;
        const int r = r0 + rowOf[i], a = ptr[r];
        if (ptr[r + 1] - a > kShort) continue;
        const unsigned long long s = sorted_at<kThreads>(lds, i);
        io.put(r, p0 + i - a, (unsigned)(s >> 12), p0 + (int)(s & 4095), p0 + i);
    }
}

template <int THREADS, typename IO>
__global__ __launch_bounds__(THREADS) void sort_long_rows_kernel(const int *__restrict__ ptr, const int *__restrict__ list, IO io)
{
    __shared__ unsigned long long lds[kPer * (THREADS + kPad)];
    const int tid = threadIdx.x, r = list[blockIdx.x], a = ptr[r], n = ptr[r + 1] - a;
    unsigned long long v[kPer];
#pragma unroll
    for (int j = 0; j < kPer; ++j) {
        const int i = j * THREADS + tid;
        v[j] = i < n ? ((unsigned long long)io.key(r, a + i) << 13) | (unsigned)i : ~0ull;
    }
    sort_workgroup<THREADS>(v, lds);
#pragma unroll
    for (int j = 0; j < kPer; ++j) {
        const int i = j * THREADS + tid;
        if (i >= n) continue;
        const unsigned long long s = sorted_at<THREADS>(lds, i);
        io.put(r, i, (unsigned)(s >> 13), a + (int)(s & 8191), a + i);
    }
}

// The classes of the rows of `ptr`: list (list_ints(entries) ints) and count (kClasses + 1, zeroed) in device memory.
inline hipError_t classify_rows(const int *ptr, int rows, int entries, int *list, int *count, hipStream_t s)
{
    if (rows > 0) hipLaunchKernelGGL(row_classes_kernel, dim3((unsigned)(((long long)rows + 255) / 256)), dim3(256), 0, s, ptr, rows, entries, list, count);
    return hipGetLastError();
}

// Every row of at most kLongest entries; `classes` is what classify_rows counted.
template <typename IO>
inline hipError_t sort_rows(const int *ptr, int rows, int entries, const int *list, const RowClasses &classes, const IO &io, hipStream_t s)
{
    if (rows <= 0 || entries <= 0) return hipSuccess;
    if (classes.n[2])
        hipLaunchKernelGGL((sort_long_rows_kernel<1024, IO>), dim3((unsigned)classes.n[2]), dim3(1024), 0, s, ptr, list + list_at(2, entries), io);
    if (classes.n[1])
        hipLaunchKernelGGL((sort_long_rows_kernel<512, IO>), dim3((unsigned)classes.n[1]), dim3(512), 0, s, ptr, list + list_at(1, entries), io);
    if (classes.n[0])
        hipLaunchKernelGGL((sort_long_rows_kernel<256, IO>), dim3((unsigned)classes.n[0]), dim3(256), 0, s, ptr, list + list_at(0, entries), io);
    hipLaunchKernelGGL(sort_short_rows_kernel<IO>, dim3((unsigned)(((long long)entries + kTile - 1) / kTile)), dim3(kThreads), 0, s, ptr, rows, io);
    return hipGetLastError();
}

}  // namespace mxs

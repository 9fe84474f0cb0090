// Transposes on the device.
//
// The reference transposes on the GPU as well -- csr2csc / csc2csr copy the matrix to the
// device, call cusparseCsr2cscEx2 and copy the result back (utilities/csr2csc.cpp:4-203), three
// times per run (test/test_autotc_spmv.cpp:1119-1238).  Here the matrix stays where it is: the
// entry point takes device arrays and leaves device arrays, so a caller that already holds the
// matrix in HBM pays no PCIe traffic.  The order inside every output line is the one the host
// transpose (mx_transpose) produces -- ascending source line, equal pairs in source order -- so
// the two are interchangeable bit for bit.
//
// A transpose is a stable sort of the entries by their index, and the lines and values travel with
// the sort.  It is made in two steps, each of which reads and writes every entry once: the entries of a tile go
// to buckets of consecutive output lines (bucket_entries_kernel), and a workgroup puts one bucket in order
// in LDS (bucket_lines_kernel).  Both are counting sorts: an entry's place among those of its digit is
// the number of lanes below it with the same digit, found with one ballot per bit of it, on top of what the waves and
// tiles before it counted -- no atomics decide an order.  In binary64 the two steps move 28 bytes an entry in and as many out, and 4 to count them
// first: 60 us at the rate of a large copy, of the 200 that the kernels take (2.4 and 2.7 TB/s).  Half of a wave's time goes into waits (for loads and
// stores, and for the rest of its workgroup between the passes over LDS), a third into its turn to issue (the ballots), 6 % into LDS.  (7.6 million entries of a power law, 700001 x 412345, binary64: 219 us;
// three passes of a radix sort over index and entry number, with the lines and values gathered at the end, 448; 2 million lines, 4.1 million output lines, binary16: 287, 1046; 12000 x 9000 with nine a line: 63, 103.)
//
// One workgroup works on a bucket; a few crowded ones are counted and put in order by as many workgroups as they have tiles (line_counts_kernel,
// line_entries_kernel), after a look by the host at which those are.  A matrix with many of them, or with more output lines than the
// buckets hold (kDigits each), takes the radix sort.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdint>
#include <cstring>
#include <string>

#include <rocprim/device/device_radix_sort.hpp>

#include "mx_device.h"
#include "mx_digits.h"
#include "mx_entry_rows.h"
#include "mx_internal.h"

namespace mxt {

using namespace mxd;

constexpr int kBlock = 256;
// Entry numbers are formed as blockIdx.x * kBlock + threadIdx.x in 32 bits: the last block must not pass 2^31.
constexpr int kMaxCount = 2147483647 - 2 * kBlock;

// ---- the two steps ------------------------------------------------------------------------
// A bucket's workgroup takes 10.5 us for every 8192 of its entries while the others are done.  A bucket with too many is crowded: its tiles are put in order by
// workgroups of their own (line_entries_kernel), which takes a look by the host at which buckets those are and four launches for each.
// That is 30 us, as long as three rounds of its own workgroup; for 8 million binary16 entries, where the others take longer, as four.  Us, binary64, n entries of which m
// name one line of many, by the bucket's own workgroup / by workgroups for its tiles / by the radix sort alone: n = 60 thousand, m = 32 thousand
// 106 / 94 / 89; 300 and 96 thousand 221 / 99 / 176; a million and 32 thousand 142 / 113 / 247; a million and 300 thousand 584 / 112 / 239; 8 million and
// 300 thousand 769 / 285 / 626.
constexpr int kCrowdedMost = 8;  // crowded buckets at most; where more have so many, they may have as many as take as long as the radix sort and the counting
inline BucketBound bucket_bound(int nnz)
{
    constexpr int low = 24576;
    return BucketBound{kCrowdedMost, low, std::max(low, std::min(30000 + nnz / 6, 75000 + nnz / 50))};
}
constexpr int kBucketsWorth = 1024;  // entries from which on the buckets are faster than a sort by one workgroup (800: 57 us, radix sort 50; 1250: 57, 59)

// An entry between the two steps, in one piece: a store of a wave goes to as many places as it has lanes, whatever a lane
// stores (line, source line and value in arrays of their own, put in order in LDS to be written side by side: 89 + 89 us
// in the two steps for 7.6 million binary64 entries, so 92 + 65).
template <typename V>
struct Moved;
template <>
struct Moved<double> {
    typedef int4 Word;
    static __device__ __forceinline__ Word pack(int line, int source, double v)
    {
        const unsigned long long u = __builtin_bit_cast(unsigned long long, v);
        return make_int4((int)(unsigned)u, (int)(unsigned)(u >> 32), source, line);
    }
    static __device__ __forceinline__ int line(const Word &w) { return w.w; }
    static __device__ __forceinline__ int source(const Word &w) { return w.z; }
    static __device__ __forceinline__ double value(const Word &w)
    {
        return __builtin_bit_cast(double, ((unsigned long long)(unsigned)w.y << 32) | (unsigned)w.x);
    }
};
template <>
struct Moved<uint16_t> {
    typedef int2 Word;
    static __device__ __forceinline__ Word pack(int line, int source, uint16_t v) { return make_int2(source, line | (int)((unsigned)v << 16)); }
    static __device__ __forceinline__ int line(const Word &w) { return w.y & 0xffff; }
    static __device__ __forceinline__ int source(const Word &w) { return w.x; }
    static __device__ __forceinline__ uint16_t value(const Word &w) { return (uint16_t)((unsigned)w.y >> 16); }
};

__device__ __forceinline__ bool refused(int flag) { return flag & (kBucketsBad | kBucketsRefused); }

// The entries of a tile to their buckets, in source order.
template <typename V>
__global__ __launch_bounds__(kThreads, 8) void bucket_entries_kernel(const int *__restrict__ ptr, const int *__restrict__ ind, const V *__restrict__ val,
                                                                     int outer, int nnz, Buckets B, int tiles, const int *__restrict__ before,
                                                                     const int *__restrict__ first, const int *__restrict__ flag,
                                                                     typename Moved<V>::Word *__restrict__ moved)
{
    __shared__ union {
        mxr::TileRowsOf<kThreads, kPer> rows;
        Digits digits;
    } U;
    __shared__ int start[kDigits];
    const int t = tile_of_block(tiles);
    if (t >= tiles || refused(flag[0])) return;
    const int t0 = t * kTile, tid = threadIdx.x, lane = tid & 63, w = tid >> 6, size = min(kTile, nnz - t0);
    mxr::tile_rows(ptr, outer, nnz, t0, U.rows);
    int row[kPer], c[kPer], at[kPer];  // (c: bucket and line)
#pragma unroll
    for (int j = 0; j < kPer; ++j) {
        const int i = w * kWave + j * 64 + lane;
        c[j] = i < size ? ind[t0 + i] : 0;
        row[j] = i < size ? U.rows.row[i] : 0;
    }
    for (int k = tid; k < B.n; k += kThreads) start[k] = first[k] + before[(size_t)t * B.n + k];
#pragma unroll
    for (int j = 0; j < kPer; ++j) {
        const int b = B.of(c[j]);
        c[j] = b | (c[j] - b * B.lines) << 16;
    }
    __syncthreads();
    place_by_digit<false>([&](int j) { return c[j] & 0xffff; }, size, B.bits, U.digits, start, (int *)nullptr, at);
    V v[kPer];
#pragma unroll
    for (int j = 0; j < kPer; ++j) v[j] = val[t0 + min(w * kWave + j * 64 + lane, size - 1)];
    __builtin_amdgcn_sched_barrier(0);  // (all values are asked for before the first is waited for)
#pragma unroll
    for (int j = 0; j < kPer; ++j)
        if (w * kWave + j * 64 + lane < size) moved[at[j]] = Moved<V>::pack(c[j] >> 16, row[j], v[j]);
}

// A bucket in order of its lines, and the pointers of its lines.  One of at most kTile entries is put in order in LDS
// and written as it comes out; a larger one takes several rounds, whose entries go behind what the rounds before left of
// their lines, each to its own place.
template <typename V>
__global__ __launch_bounds__(kThreads, 8) void bucket_lines_kernel(const typename Moved<V>::Word *__restrict__ moved, const int *__restrict__ first,
                                                                   int inner, Buckets B, const int *__restrict__ flag, int *__restrict__ tPtr,
                                                                   int *__restrict__ tInd, V *__restrict__ tVal)
{
    typedef Moved<V> M;
    __shared__ union {
        Digits digits;
        V val[kTile];
        int word[kTile];
    } U;
    __shared__ int next[kDigits], part[kWaves];
    __shared__ unsigned short start[kDigits];
    if (refused(flag[0])) return;
    const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6, b = blockIdx.x;
    const int c0 = b * B.lines, lines = min(B.lines, inner - c0), p0 = first[b], p1 = first[b + 1];
    if (b == B.n - 1 && tid == 0) tPtr[inner] = p1;
    if (p1 - p0 > flag[1]) return;  // (crowded)
    int d[kPer], at[kPer], row[kPer];
    V v[kPer];
    auto load = [&](int q, int size) {
#pragma unroll
        for (int j = 0; j < kPer; ++j) {
            const int i = w * kWave + j * 64 + lane;
            const typename M::Word e = moved[q + min(i, size - 1)];
            d[j] = M::line(e);
            row[j] = M::source(e);
            v[j] = M::value(e);
        }
    };
    if (p1 - p0 <= kTile) {
        const int size = p1 - p0;
        if (size > 0) load(p0, size);
        place_by_digit<true>([&](int j) { return d[j]; }, size, B.lineBits, U.digits, start, part, at);
        for (int c = tid; c < lines; c += kThreads) tPtr[c0 + c] = p0 + start[c];
#pragma unroll
        for (int j = 0; j < kPer; ++j)
            if (w * kWave + j * 64 + lane < size) U.word[at[j]] = row[j];
        __syncthreads();
#pragma unroll
        for (int j = 0; j < kPer; ++j)
            if (j * kThreads + tid < size) tInd[p0 + j * kThreads + tid] = U.word[j * kThreads + tid];
        __syncthreads();
#pragma unroll
        for (int j = 0; j < kPer; ++j)
            if (w * kWave + j * 64 + lane < size) U.val[at[j]] = v[j];
        __syncthreads();
#pragma unroll
        for (int j = 0; j < kPer; ++j)
            if (j * kThreads + tid < size) tVal[p0 + j * kThreads + tid] = U.val[j * kThreads + tid];
        return;
    }
    next[2 * tid] = next[2 * tid + 1] = 0;
    __syncthreads();
    // (places are unsigned here: the step past the last entry is more than an int holds where the bucket ends near 2^31)
    const unsigned end = (unsigned)p1;
    for (unsigned p = (unsigned)p0; p < end; p += kThreads) {
        const int c = p + tid < end ? M::line(moved[p + tid]) : -1, one = __builtin_amdgcn_readfirstlane(c);
        const unsigned long long same = __ballot(c == one);  // (a crowded line)
        if (one >= 0 && lane == __builtin_ctzll(same)) atomicAdd(&next[one], __popcll(same));
        if (c >= 0 && c != one) atomicAdd(&next[c], 1);
    }
    __syncthreads();
    {
        const int n0 = next[2 * tid], n1 = next[2 * tid + 1], s = p0 + sum_before(n0 + n1, part);
        next[2 * tid] = s;
        next[2 * tid + 1] = s + n0;
        if (2 * tid < lines) tPtr[c0 + 2 * tid] = s;
        if (2 * tid + 1 < lines) tPtr[c0 + 2 * tid + 1] = s + n0;
    }
    for (unsigned q = (unsigned)p0; q < end; q += kTile) {
        const int size = min(kTile, (int)(end - q));
        load((int)q, size);
        place_by_digit<true>([&](int j) { return d[j]; }, size, B.lineBits, U.digits, start, part, at);
#pragma unroll
        for (int j = 0; j < kPer; ++j) {
            if (w * kWave + j * 64 + lane >= size) continue;
            const int to = next[d[j]] + at[j] - start[d[j]];
            tInd[to] = row[j];
            tVal[to] = v[j];
        }
        __syncthreads();
        const int s0 = start[2 * tid], s1 = start[2 * tid + 1], s2 = tid + 1 < kThreads ? start[2 * tid + 2] : size;
        next[2 * tid] += s1 - s0;
        next[2 * tid + 1] += s2 - s1;
    }
}

// ---- a crowded bucket, by as many workgroups as it has tiles ----
// count[tile][line] entries
template <typename V>
__global__ __launch_bounds__(kThreads) void line_counts_kernel(const typename Moved<V>::Word *__restrict__ moved, int n, int lines, int tiles,
                                                               int *__restrict__ count)
{
    __shared__ int here[kDigits];
    const int t = tile_of_block(tiles), tid = threadIdx.x, lane = tid & 63;
    if (t >= tiles) return;
    const int t0 = t * kTile, size = min(kTile, n - t0);
    here[tid] = here[tid + kThreads] = 0;
    __syncthreads();
    for (int i = tid; i < size; i += kThreads) {
        const int c = Moved<V>::line(moved[t0 + i]), one = __builtin_amdgcn_readfirstlane(c);
        const unsigned long long same = __ballot(c == one);  // (a crowded line)
        if (lane == __builtin_ctzll(same)) atomicAdd(&here[one], __popcll(same));
        if (c != one) atomicAdd(&here[c], 1);
    }
    __syncthreads();
    for (int k = tid; k < lines; k += kThreads) count[(size_t)t * lines + k] = here[k];
}
// Every entry to its place, from the entries of its line in the tiles before (`before`) and of the lines before (`first`); the pointers of the lines.
template <typename V>
__global__ __launch_bounds__(kThreads, 8) void line_entries_kernel(const typename Moved<V>::Word *__restrict__ moved, int n, int lines, int lineBits, int tiles,
                                                                   const int *__restrict__ before, const int *__restrict__ first, int p0,
                                                                   int *__restrict__ tPtr, int *__restrict__ tInd, V *__restrict__ tVal)
{
    __shared__ Digits digits;
    __shared__ int start[kDigits];
    const int t = tile_of_block(tiles), tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
    if (t >= tiles) return;
    const int t0 = t * kTile, size = min(kTile, n - t0);
    for (int k = tid; k < lines; k += kThreads) {
        start[k] = first[k] + before[(size_t)t * lines + k];
        if (t == 0) tPtr[k] = p0 + first[k];
    }
    int d[kPer], at[kPer], row[kPer];
    V v[kPer];
#pragma unroll
    for (int j = 0; j < kPer; ++j) {
        const typename Moved<V>::Word e = moved[t0 + min(w * kWave + j * 64 + lane, size - 1)];
        d[j] = Moved<V>::line(e);
        row[j] = Moved<V>::source(e);
        v[j] = Moved<V>::value(e);
    }
    place_by_digit<false>([&](int j) { return d[j]; }, size, lineBits, digits, start, (int *)nullptr, at);
#pragma unroll
    for (int j = 0; j < kPer; ++j) {
        if (w * kWave + j * 64 + lane >= size) continue;
        tInd[at[j]] = row[j];
        tVal[at[j]] = v[j];
    }
}

// ---- the radix sort's kernels ---------------------------------------------------------------
// line[e] = r with ptr[r] <= e < ptr[r+1]; bad |= 1 where ind[e] lies outside [0, inner).
// (7 million entries in 700001 lines: 0.13 ms with a search per entry, 0.04 so)
__global__ __launch_bounds__(kBlock) void entry_lines_kernel(const int *__restrict__ ptr, const int *__restrict__ ind,
                                                             int outer, int inner, int nnz, int *__restrict__ line,
                                                             int *__restrict__ payload, int *__restrict__ bad)
{
    __shared__ mxr::TileRows T;
    const int t0 = blockIdx.x * mxr::kTile;
    mxr::tile_rows(ptr, outer, nnz, t0, T);
    bool out = false;
#pragma unroll
    for (int k = 0; k < mxr::kPer; ++k) {
        const int i = k * kBlock + threadIdx.x;
        if (i >= nnz - t0) break;
        line[t0 + i] = T.row[i];
        payload[t0 + i] = t0 + i;
        out |= (unsigned)ind[t0 + i] >= (unsigned)inner;
    }
    if (__any(out) && (threadIdx.x & 63) == 0) atomicOr(bad, 1);
}

// tPtr[c] = number of sorted keys below c, for c in [0, inner].  Thread k owns the lines
// (key[k-1], key[k]]; the thread behind the last key owns what is left, inner included.
__global__ __launch_bounds__(kBlock) void line_pointers_kernel(const int *__restrict__ key, int nnz, int inner,
                                                               int *__restrict__ tPtr)
{
    const long long k = (long long)blockIdx.x * kBlock + threadIdx.x;
    if (k > nnz) return;
    const int first = k == 0 ? 0 : key[k - 1] + 1;
    const int last = k == nnz ? inner : key[k];
    for (int c = first; c <= last; ++c) tPtr[c] = (int)k;
}

template <typename V>
__global__ __launch_bounds__(kBlock) void gather_kernel(const int *__restrict__ payload, const int *__restrict__ line,
                                                        const V *__restrict__ val, int nnz, int *__restrict__ tInd,
                                                        V *__restrict__ tVal)
{
    const int k = blockIdx.x * kBlock + threadIdx.x;
    if (k >= nnz) return;
    const int e = payload[k];
    tInd[k] = line[e];
    tVal[k] = val[e];
}

struct Scratch {
    void *p = nullptr;
    Scratch() = default;
    Scratch(const Scratch &) = delete;
    Scratch &operator=(const Scratch &) = delete;
    ~Scratch()
    {
        if (p) (void)mx::dev_free(p);
    }
};

}  // namespace mxt

#define MXT_TRY(call)                                                                                  \
    do {                                                                                               \
        hipError_t e_ = (call);                                                                        \
        if (e_ != hipSuccess) {                                                                        \
            mx::set_error(std::string("mx_transpose_device: ") + #call + ": " + hipGetErrorString(e_)); \
            return e_ == hipErrorOutOfMemory ? MX_ERR_ALLOC : MX_ERR_DEVICE;                           \
        }                                                                                              \
    } while (0)

namespace mxt {

// By buckets; *done is false, and nothing is written, where the matrix does not suit it (*checked: its indices were looked at).
template <typename V>
static int transpose_by_buckets(int outer, int inner, int nnz, const int *ptr, const int *ind, const V *val, int *tPtr, int *tInd, V *tVal,
                                bool *done, bool *checked, hipStream_t s)
{
    *done = *checked = false;
    if (!buckets_hold(inner)) return MX_OK;
    const Buckets B = make_buckets(inner, nnz);
    const BucketBound bound = bucket_bound(nnz);
    // (nor is it worth counting where the buckets have too many entries on the average: so few lines are one pass of the radix sort)
    if (nnz < kBucketsWorth || nnz / B.n > bound.high) return MX_OK;
    const int buckets = B.n, tiles = (int)(((long long)nnz + kTile - 1) / kTile);
    typedef typename Moved<V>::Word Word;
    auto al = [](size_t b) { return (b + 255) & ~(size_t)255; };
    const size_t countB = al((size_t)tiles * buckets * 4 + (size_t)tiles * 4), firstB = al((size_t)(2 * kDigits + 3) * 4);
    Scratch scratch;
    MXT_TRY(mx::dev_malloc(&scratch.p, countB + firstB + (size_t)nnz * sizeof(Word)));
    unsigned char *b = (unsigned char *)scratch.p;
    int *count = (int *)b, *bad = count + (size_t)tiles * buckets, *flag = (int *)(b + countB), *first = flag + 2, *total = first + kDigits + 1;
    Word *moved = (Word *)(b + countB + firstB);
    hipLaunchKernelGGL(bucket_counts_kernel, tile_blocks(tiles), dim3(kThreads), 0, s, ind, inner, nnz, B, tiles, count, bad);
    hipLaunchKernelGGL(bucket_offsets_kernel, dim3((unsigned)((buckets + 15) / 16)), dim3(1024), 0, s, count, buckets, tiles, total);
    hipLaunchKernelGGL(bucket_starts_kernel<true>, dim3(1), dim3(kThreads), 0, s, (const int *)total, buckets, bound, (const int *)bad, tiles,
                       first, flag);
    hipLaunchKernelGGL(bucket_entries_kernel<V>, tile_blocks(tiles), dim3(kThreads), 0, s, ptr, ind, val, outer, nnz, B, tiles, (const int *)count,
                       (const int *)first, (const int *)flag, moved);
    hipLaunchKernelGGL(bucket_lines_kernel<V>, dim3((unsigned)buckets), dim3(kThreads), 0, s, (const Word *)moved, (const int *)first, inner, B, (const int *)flag, tPtr, tInd, tVal);
    MXT_TRY(hipGetLastError());
    int got[2 + kDigits + 1];  // (flag and first)
    MXT_TRY(hipMemcpyAsync(got, flag, ((size_t)buckets + 3) * 4, hipMemcpyDeviceToHost, s));
    MXT_TRY(hipStreamSynchronize(s));
    if (got[0] & kBucketsBad) {
        mx::set_error("mx_transpose_device: index out of range");
        return MX_ERR_ARG;
    }
    *checked = true;
    *done = !(got[0] & kBucketsRefused);
    if (!(got[0] & kBucketsCrowded) || !*done) return MX_OK;
    const int *from = got + 2;
    int most = 0;
    for (int k = 0; k < buckets; ++k) most = std::max(most, from[k + 1] - from[k]);
    const size_t lineCountB = al((size_t)((most - 1) / kTile + 1) * B.lines * 4);
    Scratch crowd;
    MXT_TRY(mx::dev_malloc(&crowd.p, lineCountB + al((size_t)(2 * kDigits + 2) * 4)));
    int *lineCount = (int *)crowd.p, *lineFirst = (int *)((unsigned char *)crowd.p + lineCountB), *lineTotal = lineFirst + kDigits + 1, *unused = lineTotal + kDigits;
    for (int k = 0; k < buckets; ++k) {
        const int p0 = from[k], n = from[k + 1] - p0, c0 = k * B.lines, lines = std::min(B.lines, inner - c0), lineTiles = (n - 1) / kTile + 1;
        if (n <= got[1]) continue;
        const Word *here = moved + p0;
        hipLaunchKernelGGL(line_counts_kernel<V>, tile_blocks(lineTiles), dim3(kThreads), 0, s, here, n, lines, lineTiles, lineCount);
        hipLaunchKernelGGL(bucket_offsets_kernel, dim3((unsigned)((lines + 15) / 16)), dim3(1024), 0, s, lineCount, lines, lineTiles, lineTotal);
        hipLaunchKernelGGL(bucket_starts_kernel<false>, dim3(1), dim3(kThreads), 0, s, (const int *)lineTotal, lines, BucketBound{}, (const int *)nullptr, 0, lineFirst, unused);
        hipLaunchKernelGGL(line_entries_kernel<V>, tile_blocks(lineTiles), dim3(kThreads), 0, s, here, n, lines, B.lineBits, lineTiles, (const int *)lineCount,
                           (const int *)lineFirst, p0, tPtr + c0, tInd + p0, tVal + p0);
    }
    MXT_TRY(hipGetLastError());
    MXT_TRY(hipStreamSynchronize(s));
    return MX_OK;
}

}  // namespace mxt

extern "C" int mx_transpose_device(mx_dtype dtype, int outer, int inner, int nnz, const int *ptr_dev, const int *ind_dev,
                                   const void *val_dev, int *tPtr_dev, int *tInd_dev, void *tVal_dev, void *stream)
{
    using namespace mxt;
    if ((dtype != MX_F64 && dtype != MX_F16) || outer < 0 || inner < 0 || nnz < 0 || !ptr_dev || !tPtr_dev ||
        (nnz > 0 && (!ind_dev || !val_dev || !tInd_dev || !tVal_dev || outer == 0))) {
        mx::set_error("mx_transpose_device: bad argument");
        return MX_ERR_ARG;
    }
    if (nnz > kMaxCount || inner > kMaxCount || outer > kMaxCount) {
        mx::set_error("mx_transpose_device: more than 2^31 - 513 entries or lines");
        return MX_ERR_ARG;
    }
    hipStream_t s = (hipStream_t)stream;
    mx::MemScope scope(s);
    const int pblocks = (int)(((long long)nnz + 1 + kBlock - 1) / kBlock);
    if (nnz == 0) {
        hipLaunchKernelGGL(line_pointers_kernel, dim3(pblocks), dim3(kBlock), 0, s, (const int *)nullptr, 0, inner, tPtr_dev);
        MXT_TRY(hipGetLastError());
        MXT_TRY(hipStreamSynchronize(s));
        return MX_OK;
    }
    bool checked = false;
    {
        bool done = false;
        const int rc = dtype == MX_F64 ? transpose_by_buckets(outer, inner, nnz, ptr_dev, ind_dev, (const double *)val_dev, tPtr_dev, tInd_dev,
                                                              (double *)tVal_dev, &done, &checked, s)
                                       : transpose_by_buckets(outer, inner, nnz, ptr_dev, ind_dev, (const uint16_t *)val_dev, tPtr_dev, tInd_dev,
                                                              (uint16_t *)tVal_dev, &done, &checked, s);
        if (rc != MX_OK || done) return rc;
    }
    int bits = 1;
    while (bits < 31 && (1ll << bits) < (long long)inner) ++bits;
    // one allocation: line[nnz], payload in/out [nnz] each, keys out [nnz], flag, sort storage
    size_t sortBytes = 0;
    MXT_TRY(rocprim::radix_sort_pairs(nullptr, sortBytes, (const int *)nullptr, (int *)nullptr, (const int *)nullptr,
                                      (int *)nullptr, (size_t)nnz, 0u, (unsigned)bits, s));
    const size_t n4 = ((size_t)nnz * sizeof(int) + 255) & ~(size_t)255;
    Scratch scratch;
    MXT_TRY(mx::dev_malloc(&scratch.p, 4 * n4 + 256 + sortBytes));
    unsigned char *base = (unsigned char *)scratch.p;
    int *line = (int *)base, *payIn = (int *)(base + n4), *payOut = (int *)(base + 2 * n4), *keyOut = (int *)(base + 3 * n4);
    int *bad = (int *)(base + 4 * n4);
    void *sortTmp = base + 4 * n4 + 256;
    const int eblocks = (nnz + kBlock - 1) / kBlock;
    MXT_TRY(hipMemsetAsync(bad, 0, sizeof(int), s));
    hipLaunchKernelGGL(entry_lines_kernel, mxr::tile_grid(nnz), dim3(kBlock), 0, s, ptr_dev, ind_dev, outer, inner, nnz, line,
                       payIn, bad);
    MXT_TRY(hipGetLastError());
    // an index outside [0, inner) must not reach the pointer kernel: look before going on
    if (!checked) {
        int badHost = 0;
        MXT_TRY(hipMemcpyAsync(&badHost, bad, sizeof(int), hipMemcpyDeviceToHost, s));
        MXT_TRY(hipStreamSynchronize(s));
        if (badHost) {
            mx::set_error("mx_transpose_device: index out of range");
            return MX_ERR_ARG;
        }
    }
    MXT_TRY(rocprim::radix_sort_pairs(sortTmp, sortBytes, ind_dev, keyOut, (const int *)payIn, payOut, (size_t)nnz, 0u,
                                      (unsigned)bits, s));
    hipLaunchKernelGGL(line_pointers_kernel, dim3(pblocks), dim3(kBlock), 0, s, (const int *)keyOut, nnz, inner, tPtr_dev);
    MXT_TRY(hipGetLastError());
    if (dtype == MX_F64)
        hipLaunchKernelGGL(gather_kernel<double>, dim3(eblocks), dim3(kBlock), 0, s, (const int *)payOut, (const int *)line,
                           (const double *)val_dev, nnz, tInd_dev, (double *)tVal_dev);
    else
        hipLaunchKernelGGL(gather_kernel<uint16_t>, dim3(eblocks), dim3(kBlock), 0, s, (const int *)payOut,
                           (const int *)line, (const uint16_t *)val_dev, nnz, tInd_dev, (uint16_t *)tVal_dev);
    MXT_TRY(hipGetLastError());
    MXT_TRY(hipStreamSynchronize(s));  // the scratch is released on return
    return MX_OK;
}

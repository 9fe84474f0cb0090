// Counting sorts by one digit, shared by the kernels that transpose and those that plan (mx_transpose.hip, mx_chunks.hip).
//
// An entry's place among those of its digit is the number of lanes below it with the same digit, found with one ballot per bit
// of it, on top of what the waves and tiles before it counted: no atomics decide an order, so equal digits stay as they were.
#pragma once
#include <hip/hip_runtime.h>

#include <algorithm>

namespace mxd {

constexpr int kThreads = 1024, kPer = 8, kTile = kThreads * kPer;  // entries that a workgroup puts in order at a time
constexpr int kWaves = kThreads / 64, kWave = 64 * kPer;
constexpr int kDigitBits = 11, kDigits = 1 << kDigitBits;  // values of a digit

// The lanes of the wave whose digit is this lane's; `live` are those that have one.
__device__ __forceinline__ unsigned long long same_digit(unsigned d, int bits, unsigned long long live)
{
    unsigned lo = (unsigned)live, hi = (unsigned)(live >> 32);
#pragma unroll
    for (int k = 0; k < kDigitBits; ++k)
        if (k < bits) {
            const unsigned set = (unsigned)((int)(d << (31 - k)) >> 31);  // all bits, or none
            const unsigned long long b = __ballot(set != 0);
            lo &= ~((unsigned)b ^ set);
            hi &= ~((unsigned)(b >> 32) ^ set);
        }
    return ((unsigned long long)hi << 32) | lo;
}
__device__ __forceinline__ int lanes_below(unsigned long long m)
{
    return __builtin_amdgcn_mbcnt_hi((unsigned)(m >> 32), __builtin_amdgcn_mbcnt_lo((unsigned)m, 0));
}
// The sum of v over the threads of the workgroup before this one; `part` has room for a wave each.
__device__ __forceinline__ int sum_before(int v, int *part)
{
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    int run = v;
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
        const int o = __shfl_up(run, off);
        if (lane >= off) run += o;
    }
    if (lane == 63) part[w] = run;
    __syncthreads();
    int before = 0;
#pragma unroll
    for (int k = 0; k < kWaves; ++k)
        if (k < w) before += part[k];
    __syncthreads();
    return before + run - v;
}

// The `size` entries of a workgroup in order of their digits, equal digits in order of their numbers: entry
// i = w * kWave + j * 64 + lane belongs to thread (w, lane), digit(j) is its digit and at[j] becomes its place behind
// start[digit].  SUM: start[k] is set to the entries of the digits before k, for every k up to kDigits; otherwise it is the
// caller's.  D is free again on return.
struct Digits {
    unsigned short seen[kWaves][kDigits];
};
template <bool SUM, typename T, typename F>
__device__ __forceinline__ void place_by_digit(const F &digit, int size, int bits, Digits &D, T *__restrict__ start, int *__restrict__ part,
                                               int (&at)[kPer])
{
    const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
    for (int i = tid; i < kWaves * kDigits / 8; i += kThreads) ((int4 *)D.seen)[i] = make_int4(0, 0, 0, 0);
    __syncthreads();
    unsigned short *mine = D.seen[w];
#pragma unroll
    for (int j = 0; j < kPer; ++j) {
        const bool live = w * kWave + j * 64 + lane < size;
        const int k = digit(j);
        const unsigned long long m = same_digit((unsigned)k, bits, __ballot(live));
        const int had = live ? mine[k] : 0, below = lanes_below(m);
        // (a wave's LDS accesses happen in order; the fences keep the compiler from moving one over another)
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        if (live && below == 0) mine[k] = (unsigned short)(had + __popcll(m));
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        at[j] = had + below;
    }
    __syncthreads();
    // a thread takes two digits, side by side in a word (no sum passes kTile)
    unsigned n = 0;
#pragma unroll
    for (int k = 0; k < kWaves; ++k) {
        unsigned *word = (unsigned *)&D.seen[k][2 * tid];
        const unsigned c = *word;
        *word = n;
        n += c;
    }
    if (SUM) {
        const int n0 = (int)(n & 0xffff), n1 = (int)(n >> 16), s = sum_before(n0 + n1, part);
        start[2 * tid] = (T)s;
        start[2 * tid + 1] = (T)(s + n0);
    }
    __syncthreads();
#pragma unroll
    for (int j = 0; j < kPer; ++j) {
        const int k = digit(j);
        if (w * kWave + j * 64 + lane < size) at[j] += start[k] + mine[k];
    }
    __syncthreads();
}
static_assert(kDigits == 2 * kThreads && kTile < 65536, "two digits to a thread, counts of 16 bits");

// The tile of a workgroup: every XCD takes one stretch of the tiles, so that the pieces that follow each other in a
// bucket are written through one L2.
constexpr int kXcds = 8;
__device__ __forceinline__ int tile_of_block(int tiles)
{
    const int per = (tiles + kXcds - 1) / kXcds, k = blockIdx.x / kXcds;
    return k < per ? (int)(blockIdx.x % kXcds) * per + k : tiles;
}
inline dim3 tile_blocks(int tiles) { return dim3((unsigned)((tiles + kXcds - 1) / kXcds * kXcds)); }

// count[t][b] becomes the entries of bucket b in the tiles before t, total[b] those in all; a workgroup takes 16 buckets,
// 64 stretches of tiles of each.
static __global__ __launch_bounds__(1024) void bucket_offsets_kernel(int *__restrict__ count, int buckets, int tiles, int *__restrict__ total)
{
    __shared__ int part[64][16];
    const int k = threadIdx.x & 15, w = threadIdx.x >> 4, b = blockIdx.x * 16 + k, per = (tiles + 63) / 64;
    const int a = min(tiles, w * per), z = min(tiles, a + per);
    int sum = 0;
    if (b < buckets)
#pragma unroll 4
        for (int t = a; t < z; ++t) sum += count[(size_t)t * buckets + b];
    part[w][k] = sum;
    __syncthreads();
    if (b >= buckets) return;
    int run = 0, all = 0;
    for (int i = 0; i < 64; ++i) {
        if (i < w) run += part[i][k];
        all += part[i][k];
    }
    if (w == 0) total[b] = all;
    for (int t = a; t < z; t += 4) {
        int c[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) c[i] = t + i < z ? count[(size_t)(t + i) * buckets + b] : 0;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            if (t + i < z) count[(size_t)(t + i) * buckets + b] = run;
            run += c[i];
        }
    }
}
// How many entries a bucket may have for one workgroup to work on it.
struct BucketBound {
    int few, low, high;  // `low`, or `high` where more than `few` buckets have more than that
};
enum { kBucketsBad = 1, kBucketsCrowded = 2, kBucketsRefused = 4 };
// first[b] = entries of the buckets before b, first[buckets] = all.  flag[0]: kBucketsBad when a tile is bad; with a bound, flag[1] = the one that
// holds, kBucketsCrowded when some bucket has more than that, kBucketsRefused as well when more than `few` have.
template <bool BOUND>
static __global__ __launch_bounds__(kThreads) void bucket_starts_kernel(const int *__restrict__ total, int buckets, BucketBound bound,
                                                                        const int *__restrict__ bad, int tiles, int *__restrict__ first, int *__restrict__ flag)
{
    __shared__ int part[kWaves];
    const int b = 2 * threadIdx.x, n0 = b < buckets ? total[b] : 0, n1 = b + 1 < buckets ? total[b + 1] : 0, at = sum_before(n0 + n1, part);
    if (b <= buckets) first[b] = at;
    if (b + 1 <= buckets) first[b + 1] = at + n0;
    if (b + 2 == buckets) first[buckets] = at + n0 + n1;
    bool out = false;
    for (int t = threadIdx.x; t < tiles; t += kThreads) out |= bad[t] != 0;
    out = __syncthreads_or(out);
    int crowded = 0;
    if (BOUND) {
        auto above = [&](int m) { return __syncthreads_count(n0 > m) + __syncthreads_count(n1 > m); };
        if (__syncthreads_or(max(n0, n1) > bound.low)) crowded = above(bound.low);
        const bool many = crowded > bound.few;
        if (many) crowded = above(bound.high);
        if (b == 0) flag[1] = many ? bound.high : bound.low;
    }
    if (b == 0) flag[0] = (out ? kBucketsBad : 0) + (crowded > 0 ? kBucketsCrowded : 0) + (crowded > bound.few ? kBucketsRefused : 0);
}

// ---- buckets of consecutive lines (columns): entries by line in two steps, bucket and line inside it ----
constexpr int kBucketMean = 6800;     // entries of a bucket on average: nearly all then have at most kTile
constexpr int kBucketsLeast = 64;     // but not so few buckets that most of the device has none
// Buckets of `lines` output lines.  c / lines as a product: exact for c < kDigits * lines with lines <= kDigits, since the
// error of `inverse`, below one, times c stays below 2^42 / lines.
struct Buckets {
    int n, bits, lines, lineBits;
    unsigned long long inverse;  // 2^42 / lines, rounded up
    __device__ __forceinline__ int of(int c) const { return (int)(((unsigned long long)(unsigned)c * inverse) >> 42); }
};

// count[tile][bucket] entries; bad[tile]: an index lies outside [0, inner)
static __global__ __launch_bounds__(kThreads) void bucket_counts_kernel(const int *__restrict__ ind, int inner, int nnz, Buckets B, int tiles,
                                                                 int *__restrict__ count, int *__restrict__ bad)
{
    __shared__ int here[kDigits];
    const int t = tile_of_block(tiles);
    if (t >= tiles) return;
    const int t0 = t * kTile, tid = threadIdx.x, lane = tid & 63;
    here[tid] = here[tid + kThreads] = 0;
    __syncthreads();
    int b[kPer];
    bool out = false;
#pragma unroll
    for (int j = 0; j < kPer; ++j) {
        const int i = j * kThreads + tid;
        b[j] = -1;
        if (i >= nnz - t0) continue;
        const int c = ind[t0 + i];
        if ((unsigned)c < (unsigned)inner) b[j] = B.of(c);
        else out = true;
    }
    // (neighbours often share a bucket, and an atomic takes as long as lanes want the same word: the first lane's bucket is counted at once)
#pragma unroll
    for (int j = 0; j < kPer; ++j) {
        const int first = __builtin_amdgcn_readfirstlane(b[j]);
        const unsigned long long same = __ballot(b[j] == first);
        if (first >= 0 && lane == __builtin_ctzll(same)) atomicAdd(&here[first], __popcll(same));
        if (b[j] >= 0 && b[j] != first) atomicAdd(&here[b[j]], 1);
    }
    out = __syncthreads_or(out);
    if (tid == 0) bad[t] = out;
    for (int k = tid; k < B.n; k += kThreads) count[(size_t)t * B.n + k] = here[k];
}

inline bool buckets_hold(int lines) { return lines >= 1 && lines <= kDigits * kDigits; }
inline Buckets make_buckets(int inner, int nnz)
{
    Buckets B;
    const long long mean = ((long long)nnz + kBucketMean - 1) / kBucketMean, wide = ((long long)inner + kDigits - 1) / kDigits;
    B.n = (int)std::min<long long>(kDigits, std::max<long long>(kBucketsLeast, std::max(mean, wide)));
    B.lines = (inner + B.n - 1) / B.n;
    B.n = (inner + B.lines - 1) / B.lines;
    B.bits = B.lineBits = 0;
    while ((1 << B.bits) < B.n) ++B.bits;
    while ((1 << B.lineBits) < B.lines) ++B.lineBits;
    B.inverse = ((1ull << 42) + B.lines - 1) / B.lines;
    return B;
}

}  // namespace mxd

// Device side of the preprocessing: the two selections of the cascaded extraction (which columns, then which rows, are
// dense), the split by them and the tile encoding.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdint>
#include <cstring>
#include <string>
#include <vector>

#include <rocprim/device/device_radix_sort.hpp>
#include <rocprim/device/device_scan.hpp>

#include "mx_device.h"
#include "mx_digits.h"
#include "mx_entry_rows.h"
#include "mx_internal.h"
#include "mx_row_sort.h"

namespace mxp {

constexpr int kBlock = 256;
// Entry numbers are formed as blockIdx.x * kBlock + threadIdx.x in 32 bits: the last block must not pass 2^31.
constexpr int kMaxCount = 2147483647 - 2 * kBlock;

// ---- selection ---------------------------------------------------------------------------
// cnt[ind[e]] += 1 for every entry (integer atomics: the result does not depend on the order).
__global__ __launch_bounds__(kBlock) void index_histogram_kernel(const int *__restrict__ ind, int nnz, int inner,
                                                                 int *__restrict__ cnt, int *__restrict__ bad)
{
    const int e = blockIdx.x * kBlock + threadIdx.x;
    if (e >= nnz) return;
    const int c = ind[e];
    if ((unsigned)c >= (unsigned)inner) atomicOr(bad, 1);
    else atomicAdd(&cnt[c], 1);
}

constexpr int kBucketCounts = 1 << 21;  // entries from which on the two steps are the faster way (atomics 28 us a million; so 58 us for 2.2 million with
                                        // what five launches take, 68 for 4.3)
// The same through buckets of columns: the entries' places in their buckets, in any order, then the columns of a bucket counted in LDS.
// (Atomics on memory: 330 us for 15.8 million entries in a million columns; so 120.)
__global__ __launch_bounds__(mxd::kThreads) void bucket_columns_kernel(const int *__restrict__ ind, int nnz, int inner, mxd::Buckets B, int tiles,
                                                                       const int *__restrict__ before, const int *__restrict__ first,
                                                                       unsigned short *__restrict__ column)
{
    __shared__ int next[mxd::kDigits];
    const int t = mxd::tile_of_block(tiles), tid = threadIdx.x;
    if (t >= tiles) return;
    const int t0 = t * mxd::kTile;
    for (int k = tid; k < B.n; k += mxd::kThreads) next[k] = first[k] + before[(size_t)t * B.n + k];
    __syncthreads();
    int c[mxd::kPer];
#pragma unroll
    for (int j = 0; j < mxd::kPer; ++j) c[j] = ind[min(t0 + j * mxd::kThreads + tid, nnz - 1)];
#pragma unroll
    for (int j = 0; j < mxd::kPer; ++j) {
        if (j * mxd::kThreads + tid >= nnz - t0 || (unsigned)c[j] >= (unsigned)inner) continue;
        const int b = B.of(c[j]);
        column[atomicAdd(&next[b], 1)] = (unsigned short)(c[j] - b * B.lines);
    }
}
__global__ __launch_bounds__(mxd::kThreads) void count_columns_kernel(const unsigned short *__restrict__ column, const int *__restrict__ first, int inner,
                                                                      mxd::Buckets B, int *__restrict__ cnt)
{
    __shared__ int here[mxd::kDigits];
    const int b = blockIdx.x, tid = threadIdx.x, lane = tid & 63, p0 = first[b], p1 = first[b + 1], c0 = b * B.lines, lines = min(B.lines, inner - c0);
    for (int k = tid; k < lines; k += mxd::kThreads) here[k] = 0;
    __syncthreads();
    for (int p = mx::next_of(p0, p1, tid); p < p1; p = mx::next_of(p, p1, mxd::kThreads)) {
        const int c = column[p], one = __builtin_amdgcn_readfirstlane(c);
        const unsigned long long same = __ballot(c == one);  // (a crowded column)
        if (lane == __builtin_ctzll(same)) atomicAdd(&here[one], __popcll(same));
        if (c != one) atomicAdd(&here[c], 1);
    }
    __syncthreads();
    for (int k = tid; k < lines; k += mxd::kThreads) cnt[c0 + k] = here[k];
}

// bad |= bit where v[i] lies outside [0, lim): the index arrays of a caller are looked at before a
// kernel uses them as addresses.
__global__ __launch_bounds__(kBlock) void range_check_kernel(const int *__restrict__ v, int n, int lim, int bit,
                                                             int *__restrict__ bad)
{
    const int i = blockIdx.x * kBlock + threadIdx.x;
    if (i < n && (unsigned)v[i] >= (unsigned)lim) atomicOr(bad, bit);
}
// bad |= bit unless ptr[0] == 0, ptr[n] == total and ptr never falls.
__global__ __launch_bounds__(kBlock) void pointer_check_kernel(const int *__restrict__ ptr, int n, int total, int bit,
                                                               int *__restrict__ bad)
{
    const int i = blockIdx.x * kBlock + threadIdx.x;
    if (i > n) return;
    const int p = ptr[i];
    if ((i == 0 && p != 0) || (i == n && p != total) || (i < n && ptr[i + 1] < p) || p < 0 || p > total) atomicOr(bad, bit);
}

// most[0] = the highest of cnt [0, n), most[1] = the longest of the rows (both zeroed before)
__global__ __launch_bounds__(kBlock) void highest_kernel(const int *__restrict__ cnt, int n, const int *__restrict__ rowPtr, int rows, int *__restrict__ most)
{
    __shared__ int a, b;
    if (threadIdx.x == 0) a = b = 0;
    __syncthreads();
    int c = 0, l = 0;
    const long long step = (long long)gridDim.x * kBlock;
#pragma unroll 4
    for (long long i = (long long)blockIdx.x * kBlock + threadIdx.x; i < n; i += step) c = max(c, cnt[i]);
#pragma unroll 4
    for (long long r = (long long)blockIdx.x * kBlock + threadIdx.x; r < rows; r += step) l = max(l, rowPtr[r + 1] - rowPtr[r]);
    atomicMax(&a, c);
    atomicMax(&b, l);
    __syncthreads();
    if (threadIdx.x == 0) {
        atomicMax(&most[0], a);
        atomicMax(&most[1], b);
    }
}

// ---- lines by count, the highest first, those of one count ascending: a counting sort, eleven bits of `most - count` at a time.
// (Two orders of a million lines, counts up to some thousands: a stable radix sort of 32-bit counts, which rocPRIM makes a merge sort of twenty launches of at this size,
// 390 us; so 100.)
struct CountDigit {
    const int *cnt, *before;  // `before`: the order so far, null for the lines as they are numbered
    int most, shift;
    __device__ __forceinline__ int line(int i) const { return before ? before[i] : i; }
    __device__ __forceinline__ int operator()(int i) const { return (max(most - cnt[line(i)], 0) >> shift) & (mxd::kDigits - 1); }
};
__global__ __launch_bounds__(mxd::kThreads) void count_digits_kernel(CountDigit digit, int n, int values, int tiles, int *__restrict__ count)
{
    __shared__ int here[mxd::kDigits];
    const int t = mxd::tile_of_block(tiles), tid = threadIdx.x;
    if (t >= tiles) return;
    for (int k = tid; k < values; k += mxd::kThreads) here[k] = 0;
    __syncthreads();
    for (int i = tid; i < mxd::kTile && t * mxd::kTile + i < n; i += mxd::kThreads) {
        const int d = digit(t * mxd::kTile + i), one = __builtin_amdgcn_readfirstlane(d);
        const unsigned long long same = __ballot(d == one);  // (most lines have a count like their neighbours')
        if ((tid & 63) == __builtin_ctzll(same)) atomicAdd(&here[one], __popcll(same));
        if (d != one) atomicAdd(&here[d], 1);
    }
    __syncthreads();
    for (int k = tid; k < values; k += mxd::kThreads) count[(size_t)t * values + k] = here[k];
}
// ONE: all lines are a single tile, whose digits the workgroup counts itself (nothing before it is read).
template <bool ONE>
__global__ __launch_bounds__(mxd::kThreads, 8) void order_digits_kernel(CountDigit digit, int n, int values, int bits, int tiles,
                                                                        const int *__restrict__ before, const int *__restrict__ first,
                                                                        int *__restrict__ order, int *__restrict__ sortedCnt)
{
    using namespace mxd;
    __shared__ Digits digits;
    __shared__ int start[kDigits], part[kWaves];
    const int t = ONE ? 0 : tile_of_block(tiles), tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
    if (t >= tiles) return;
    const int t0 = t * kTile, size = min(kTile, n - t0);
    if (!ONE)
        for (int k = tid; k < values; k += kThreads) start[k] = first[k] + before[(size_t)t * values + k];
    int d[kPer], at[kPer];
#pragma unroll
    for (int j = 0; j < kPer; ++j) d[j] = digit(t0 + min(w * kWave + j * 64 + lane, size - 1));
    place_by_digit<ONE>([&](int j) { return d[j]; }, size, bits, digits, start, part, at);
#pragma unroll
    for (int j = 0; j < kPer; ++j) {
        const int i = w * kWave + j * 64 + lane;
        if (i >= size) continue;
        const int line = digit.line(t0 + i);
        order[at[j]] = line;
        sortedCnt[at[j]] = digit.cnt[line];
    }
}

// The shortest prefix of the sorted counts whose sum reaches `target`, from their running sums:
// res[0] = its length (stays -1 when the target is out of reach), res[1] = its sum; res[2], res[3]
// = number and sum of the counts that are not zero (what an unreachable target selects).
__global__ __launch_bounds__(kBlock) void prefix_reach_kernel(const int *__restrict__ sortedCnt, const int *__restrict__ run,
                                                              int n, int target, int *__restrict__ res)
{
    const int i = blockIdx.x * kBlock + threadIdx.x;
    if (i >= n) return;
    const int s = run[i], prev = i ? run[i - 1] : 0;
    if (s >= target && (i == 0 || prev < target)) {
        res[0] = i + 1;
        res[1] = s;
    }
    if (sortedCnt[i] > 0 && (i == n - 1 || sortedCnt[i + 1] == 0)) {
        res[2] = i + 1;
        res[3] = s;
    }
}

// dense[order[i]] = 1 for the first k lines of the order
__global__ __launch_bounds__(kBlock) void mark_selected_kernel(const int *__restrict__ order, int k, unsigned char *__restrict__ dense)
{
    const int i = blockIdx.x * kBlock + threadIdx.x;
    if (i < k) dense[order[i]] = 1;
}

// rcnt[r] = entries of row r in selected columns
__global__ __launch_bounds__(kBlock) void dense_row_counts_kernel(const int *__restrict__ rowPtr, const int *__restrict__ col,
                                                                  const unsigned char *__restrict__ dense, int rows, int nnz,
                                                                  int *__restrict__ rcnt)
{
    __shared__ mxr::TileRows T;
    const int t0 = blockIdx.x * mxr::kTile, lane = threadIdx.x & 63;
    mxr::tile_rows(rowPtr, rows, nnz, t0, T);
#pragma unroll
    for (int k = 0; k < mxr::kPer; ++k) {
        // The lanes of a wave hold consecutive entries, so their rows ascend: the first lane of every run
        // of equal rows adds the run's count in one atomic (a row of thousands of entries would otherwise
        // take thousands of atomics on one address).
        const int i = k * kBlock + threadIdx.x;
        const bool in = i < nnz - t0;
        const int r = in ? T.row[i] : -1;
        const bool d = in && dense[col[t0 + i]];
        const int rPrev = __shfl_up(r, 1);
        const unsigned long long heads = __ballot(lane == 0 || r != rPrev), hits = __ballot(d);
        if (!in || !((heads >> lane) & 1)) continue;
        const unsigned long long above = lane == 63 ? 0ull : heads >> (lane + 1);
        const int next = above ? lane + 1 + __builtin_ctzll(above) : 64;
        const unsigned long long run = (next == 64 ? ~0ull : (1ull << next) - 1) & ~((1ull << lane) - 1);
        const int c = __popcll(hits & run);
        if (c) atomicAdd(&rcnt[r], c);
    }
}

// ---- split --------------------------------------------------------------------------------
// rank[order[i]] = i for the first k lines of the order
__global__ __launch_bounds__(kBlock) void scatter_rank_kernel(const int *__restrict__ order, int k, int *__restrict__ rank)
{
    const int i = blockIdx.x * kBlock + threadIdx.x;
    if (i < k) rank[order[i]] = i;
}

// notSel[c] = 1 where the column was not selected (input of the running count that numbers them)
__global__ __launch_bounds__(kBlock) void not_selected_kernel(const unsigned char *__restrict__ dense, int cols, int *__restrict__ notSel)
{
    const int c = blockIdx.x * kBlock + threadIdx.x;
    if (c <= cols) notSel[c] = c < cols ? !dense[c] : 0;
}

// new column id of an unselected column: dCols + its position among the unselected, ascending
__global__ __launch_bounds__(kBlock) void sparse_columns_kernel(const unsigned char *__restrict__ dense, const int *__restrict__ pos,
                                                                int cols, int dCols, int *__restrict__ newCol)
{
    const int c = blockIdx.x * kBlock + threadIdx.x;
    if (c < cols && !dense[c]) newCol[c] = dCols + pos[c];
}

// lengths of the residual's rows (entries in unselected columns, plus those in selected columns
// when the row itself was not selected) and of A_dd's rows (rank order); one more element, zero,
// so that a running count over n + 1 elements ends with the total
__global__ __launch_bounds__(kBlock) void split_lengths_kernel(const int *__restrict__ rowPtr, const int *__restrict__ rcnt,
                                                               const int *__restrict__ rowRank, const int *__restrict__ rowOrder,
                                                               int rows, int dRows, int *__restrict__ cdLen, int *__restrict__ ddLen)
{
    const int r = blockIdx.x * kBlock + threadIdx.x;
    if (r <= rows) cdLen[r] = r < rows ? (rowPtr[r + 1] - rowPtr[r] - rcnt[r]) + (rowRank[r] < 0 ? rcnt[r] : 0) : 0;
    if (r <= dRows) ddLen[r] = r < dRows ? rcnt[rowOrder[r]] : 0;
}

// Sort key of an entry: [which matrix][its row there][residual only: selected column?][new column].
// A_dd (matrix 0) sorts in front of the residual (matrix 1); inside a residual row the entries in
// unselected columns come first, then those in selected ones; equal keys keep source order.
// (Only for matrices with rows too long to be put in order by a workgroup; SplitRows is the other way.)
__global__ __launch_bounds__(kBlock) void split_keys_kernel(const int *__restrict__ rowPtr, const int *__restrict__ col,
                                                            const int *__restrict__ newCol, const int *__restrict__ rowRank,
                                                            int rows, int nnz, int dCols, int colBits, int rowBits,
                                                            unsigned long long *__restrict__ key, int *__restrict__ payload)
{
    __shared__ mxr::TileRows T;
    const int t0 = blockIdx.x * mxr::kTile;
    mxr::tile_rows(rowPtr, rows, nnz, t0, T);
#pragma unroll
    for (int j = 0; j < mxr::kPer; ++j) {
        const int i = j * kBlock + threadIdx.x, e = t0 + i;
        if (i >= nnz - t0) break;
        const int r = T.row[i], nc = newCol[col[e]], rank = rowRank[r];
        const bool sel = nc < dCols;
        unsigned long long k;
        if (sel && rank >= 0) k = ((unsigned long long)rank << (colBits + 1)) | (unsigned long long)nc;
        else
            k = (1ull << (rowBits + colBits + 1)) | ((unsigned long long)r << (colBits + 1)) |
                ((unsigned long long)sel << colBits) | (unsigned long long)nc;
        key[e] = k;
        payload[e] = e;
    }
}

// The split of a row inside its workgroup: by {selected column?, new column}, so that the entries in unselected columns
// come first; those behind them are A_dd's where the row was selected, too.
// (15.8 million binary16 entries in a million rows: keys, radix sort and gather 1.31 ms, so 0.44)
template <typename V>
struct SplitRows {
    const int *ptr, *col, *newCol, *rowRank, *rcnt, *ddPtr, *cdPtr;
    const V *val;
    int dCols, colBits;
    int *ddInd;
    V *ddVal;
    int *cdInd;
    V *cdVal;
    __device__ __forceinline__ unsigned key(int, int e) const
    {
        const int nc = newCol[col[e]];
        return ((unsigned)(nc < dCols) << colBits) | (unsigned)nc;
    }
    __device__ __forceinline__ void put(int r, int place, unsigned key, int e, int) const
    {
        const int nc = (int)(key & ((1u << colBits) - 1)), rank = rowRank[r], rest = ptr[r + 1] - ptr[r] - rcnt[r];
        const V v = val[e];
        if (rank >= 0 && place >= rest) {
            const int at = ddPtr[rank] + place - rest;
            ddInd[at] = nc;
            ddVal[at] = v;
        } else {
            const int at = cdPtr[r] + place;
            cdInd[at] = nc;
            cdVal[at] = v;
        }
    }
};

template <typename V>
__global__ __launch_bounds__(kBlock) void split_gather_kernel(const unsigned long long *__restrict__ key, const int *__restrict__ payload,
                                                              const V *__restrict__ val, int nnz, int nDD, int colBits,
                                                              int *__restrict__ ddInd, V *__restrict__ ddVal,
                                                              int *__restrict__ cdInd, V *__restrict__ cdVal)
{
    const int k = blockIdx.x * kBlock + threadIdx.x;
    if (k >= nnz) return;
    const int nc = (int)(key[k] & ((1ull << colBits) - 1));
    const V v = val[payload[k]];
    if (k < nDD) {
        ddInd[k] = nc;
        ddVal[k] = v;
    } else {
        cdInd[k - nDD] = nc;
        cdVal[k - nDD] = v;
    }
}

// ---- tile encoding ------------------------------------------------------------------------
// first[w] = where the entries of chunk w begin
__global__ __launch_bounds__(kBlock) void chunk_starts_kernel(const int *__restrict__ ddRowPtr, int dRows, int chunkNum, int *__restrict__ first)
{
    const int w = blockIdx.x * kBlock + threadIdx.x;
    if (w <= chunkNum) first[w] = ddRowPtr[min(w * mx::kFragM, dRows)];
}

// reach[0] = where the last chunk ends that is too long for a workgroup, *chunks = the chunks up to that one
__global__ __launch_bounds__(kBlock) void long_chunks_kernel(const int *__restrict__ first, int chunkNum, int *__restrict__ reach,
                                                            int *__restrict__ chunks)
{
    const int w = blockIdx.x * kBlock + threadIdx.x;
    const bool big = w < chunkNum && first[w + 1] - first[w] > mxs::kLongest;
    const unsigned long long m = __ballot(big);
    if (m && (threadIdx.x & 63) == 63 - __builtin_clzll(m)) {
        atomicMax(reach, first[w + 1]);
        atomicMax(chunks, w + 1);
    }
}

// key = [chunk of the entry's row][column], payload = the entry, for the first n entries of A_dd: those of the chunks up to
// the last one that a workgroup has no room for.  (A_dd's rows stand in order of their length, so these are few chunks.)
__global__ __launch_bounds__(kBlock) void tile_keys_kernel(const int *__restrict__ first, const int *__restrict__ ddCol,
                                                           int chunkNum, int n, int colBits, unsigned long long *__restrict__ key,
                                                           int *__restrict__ payload)
{
    __shared__ mxr::TileRows T;
    const int t0 = blockIdx.x * mxr::kTile;
    mxr::tile_rows(first, chunkNum, n, t0, T);
#pragma unroll
    for (int j = 0; j < mxr::kPer; ++j) {
        const int i = j * kBlock + threadIdx.x, e = t0 + i;
        if (i >= n - t0) break;
        key[e] = ((unsigned long long)T.row[i] << colBits) | (unsigned long long)ddCol[e];
        payload[e] = e;
    }
}

// The same order for the chunks that a workgroup has room for.
// (15.8 million entries, of which 5.6 lie in chunks up to the last of more than 8192: keys and radix sort 1.05 ms, so 0.69, 0.38 of them for those 5.6)
struct ChunkColumns {
    const int *ddCol;
    int colBits;
    unsigned long long *keyOut;
    int *payload;
    __device__ __forceinline__ unsigned key(int, int e) const { return (unsigned)ddCol[e]; }
    __device__ __forceinline__ void put(int chunk, int, unsigned col, int e, int k) const
    {
        keyOut[k] = ((unsigned long long)(unsigned)chunk << colBits) | col;
        payload[k] = e;
    }
};

// head[k] = 1 where sorted position k holds the first occurrence of its (chunk, column)
__global__ __launch_bounds__(kBlock) void tile_heads_kernel(const unsigned long long *__restrict__ key, int n, int *__restrict__ head)
{
    const int k = blockIdx.x * kBlock + threadIdx.x;
    if (k < n) head[k] = k == 0 || key[k] != key[k - 1];
}

// frags[w] = ceil(distinct columns of chunk w / fragK); one more element, zero.  The entries of
// chunk w sit at sorted positions [a, b) = ddRowPtr[8w] .. ddRowPtr[min(8w + 8, dRows)], and `run`
// is the inclusive running count of the heads.
__global__ __launch_bounds__(kBlock) void tile_chunk_frags_kernel(const int *__restrict__ ddRowPtr, const int *__restrict__ run,
                                                                  int dRows, int chunkNum, int fragK, int *__restrict__ frags)
{
    const int w = blockIdx.x * kBlock + threadIdx.x;
    if (w > chunkNum) return;
    int f = 0;
    if (w < chunkNum) {
        const int a = ddRowPtr[w * mx::kFragM], b = ddRowPtr[min(w * mx::kFragM + mx::kFragM, dRows)];
        if (b > a) f = (run[b - 1] - run[a] + 1 + fragK - 1) / fragK;
    }
    frags[w] = f;
}

// Per sorted position: the rank of its column inside its chunk (ecr) goes back to the entry; a
// head also writes its column into the chunk's list; every entry sets its bit.
__global__ __launch_bounds__(kBlock) void tile_rank_kernel(const unsigned long long *__restrict__ key, const int *__restrict__ payload,
                                                           const int *__restrict__ head, const int *__restrict__ run,
                                                           const int *__restrict__ ddRowPtr, const int *__restrict__ chunkPtr, int dRows,
                                                           int n, int colBits, int fragK, int *__restrict__ ecr, int *__restrict__ atox,
                                                           unsigned long long *__restrict__ bits)
{
    const int k = blockIdx.x * kBlock + threadIdx.x, lane = threadIdx.x & 63;
    int f = -1;
    unsigned long long v = 0;
    if (k < n) {
        const int w = (int)(key[k] >> colBits), c = (int)(key[k] & ((1ull << colBits) - 1));
        const int rank = run[k] - run[ddRowPtr[w * mx::kFragM]];
        const int e = payload[k];
        ecr[e] = rank;
        const int f0 = chunkPtr[w];
        if (head[k]) atox[(size_t)f0 * fragK + rank] = c;
        int r = 0;  // the row inside the chunk
#pragma unroll
        for (int i = 1; i < mx::kFragM; ++i) r += ddRowPtr[min(w * mx::kFragM + i, dRows)] <= e;
        f = f0 + rank / fragK;
        v = 1ull << (r * fragK + rank % fragK);
    }
    // Sorted positions ascend by (chunk, column), so the fragments of a wave's lanes ascend too: the
    // bits of every run of equal fragments are gathered at its first lane, which issues one atomic.
    const int fPrev = __shfl_up(f, 1);
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
        const unsigned long long o = __shfl_down(v, off);
        const int fo = __shfl_down(f, off);
        if (lane + off < 64 && fo == f) v |= o;
    }
    if (f >= 0 && (lane == 0 || f != fPrev)) atomicOr(&bits[f], v);
}

// count[f] = set bits of fragment f; one more element, zero
__global__ __launch_bounds__(kBlock) void tile_popcount_kernel(const unsigned long long *__restrict__ bits, int nf, int *__restrict__ count)
{
    const int f = blockIdx.x * kBlock + threadIdx.x;
    if (f <= nf) count[f] = f < nf ? __popcll(bits[f]) : 0;
}

// Values of a fragment in ascending bit order: an entry's place is the number of set bits below
// its own.  Of entries that name the same row and column (neighbours in the sorted row) the last
// one is kept.
template <typename V>
__global__ __launch_bounds__(kBlock) void tile_values_kernel(const int *__restrict__ ddRowPtr, const int *__restrict__ ddCol,
                                                             const V *__restrict__ ddVal, const int *__restrict__ ecr,
                                                             const int *__restrict__ chunkPtr, const int *__restrict__ fragPtr,
                                                             const unsigned long long *__restrict__ bits, int dRows, int n, int fragK,
                                                             V *__restrict__ tcVal)
{
    __shared__ mxr::TileRows T;
    const int t0 = blockIdx.x * mxr::kTile;
    mxr::tile_rows(ddRowPtr, dRows, n, t0, T);
#pragma unroll
    for (int j = 0; j < mxr::kPer; ++j) {
        const int k = j * kBlock + threadIdx.x, e = t0 + k;
        if (k >= n - t0) break;
        const int i = T.row[k];
        if (e + 1 < ddRowPtr[i + 1] && ddCol[e + 1] == ddCol[e]) continue;  // a later twin wins
        const int w = i / mx::kFragM, rank = ecr[e], f = chunkPtr[w] + rank / fragK;
        const int bit = (i - w * mx::kFragM) * fragK + rank % fragK;
        tcVal[fragPtr[f] + __popcll(bits[f] & ((1ull << bit) - 1))] = ddVal[e];
    }
}

__global__ __launch_bounds__(kBlock) void narrow_bits_kernel(const unsigned long long *__restrict__ bits, int nf, unsigned *__restrict__ out)
{
    const int f = blockIdx.x * kBlock + threadIdx.x;
    if (f < nf) out[f] = (unsigned)bits[f];
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

}  // namespace mxp

// `who` is the name of the entry point the enclosing function works for
#define MXP_TRY(call)                                                                       \
    do {                                                                                    \
        hipError_t e_ = (call);                                                             \
        if (e_ != hipSuccess) {                                                             \
            mx::set_error(std::string(who) + ": " + #call + ": " + hipGetErrorString(e_)); \
            return e_ == hipErrorOutOfMemory ? MX_ERR_ALLOC : MX_ERR_DEVICE;                \
        }                                                                                   \
    } while (0)

namespace mxp {

// order[0..n) = the lines by count descending, ties by ascending line; then the prefix that reaches `target`.
// cnt, order: device arrays of n, no count above `most`; work: 3 n ints + 4, digitTmp: digit_bytes(n); returns the
// prefix length and its sum.
static size_t digit_bytes(size_t n)
{
    return ((n + mxd::kTile - 1) / mxd::kTile * mxd::kDigits + 2 * mxd::kDigits + 64) * sizeof(int);
}
static int order_and_reach(const int *cnt, int n, int most, int target, int *order, int *work, int *digitTmp,
                           void *scanTmp, size_t scanBytes, hipStream_t s, int *len, int *sum)
{
    static const char who[] = "mx_select_device";
    *len = 0;
    *sum = 0;
    if (n == 0) return MX_OK;
    int *other = work, *sortedCnt = work + n, *run = work + 2 * (size_t)n, *res = work + 3 * (size_t)n;
    const int blocks = (n + kBlock - 1) / kBlock, tiles = (int)(((long long)n + mxd::kTile - 1) / mxd::kTile);
    int *total = digitTmp, *first = total + mxd::kDigits, *flag = first + mxd::kDigits + 1, *count = total + 2 * mxd::kDigits + 64;
    int passes = 1;
    while (passes < 3 && (most >> (mxd::kDigitBits * passes)) > 0) ++passes;
    const int *before = nullptr;
    for (int p = 0; p < passes; ++p) {
        int *out = (passes - 1 - p) % 2 == 0 ? order : other;  // (the last one writes `order`)
        const int shift = p * mxd::kDigitBits, values = std::min(mxd::kDigits, (most >> shift) + 1);
        int bits = 0;
        while ((1 << bits) < values) ++bits;
        const CountDigit digit{cnt, before, most, shift};
        if (tiles == 1) {  // (one launch instead of four: the partition of 2000 entries 498 us, 544 with four)
            hipLaunchKernelGGL(order_digits_kernel<true>, dim3(1), dim3(mxd::kThreads), 0, s, digit, n, values, bits, 1, (const int *)nullptr, (const int *)nullptr, out,
                               sortedCnt);
            before = out;
            continue;
        }
        hipLaunchKernelGGL(count_digits_kernel, mxd::tile_blocks(tiles), dim3(mxd::kThreads), 0, s, digit, n, values, tiles, count);
        hipLaunchKernelGGL(mxd::bucket_offsets_kernel, dim3((unsigned)((values + 15) / 16)), dim3(1024), 0, s, count, values, tiles, total);
        hipLaunchKernelGGL(mxd::bucket_starts_kernel<false>, dim3(1), dim3(mxd::kThreads), 0, s, (const int *)total, values, mxd::BucketBound{}, (const int *)nullptr, 0, first, flag);
        hipLaunchKernelGGL(order_digits_kernel<false>, mxd::tile_blocks(tiles), dim3(mxd::kThreads), 0, s, digit, n, values, bits, tiles, (const int *)count,
                           (const int *)first, out, sortedCnt);
        before = out;
    }
    MXP_TRY(hipGetLastError());
    MXP_TRY(rocprim::inclusive_scan(scanTmp, scanBytes, (const int *)sortedCnt, run, (size_t)n, rocprim::plus<int>(), s));
    const int init[4] = {-1, 0, 0, 0};
    MXP_TRY(hipMemcpyAsync(res, init, sizeof(init), hipMemcpyHostToDevice, s));
    hipLaunchKernelGGL(prefix_reach_kernel, dim3(blocks), dim3(kBlock), 0, s, (const int *)sortedCnt, (const int *)run, n,
                       target, res);
    MXP_TRY(hipGetLastError());
    int got[4];
    MXP_TRY(hipMemcpyAsync(got, res, sizeof(got), hipMemcpyDeviceToHost, s));
    MXP_TRY(hipStreamSynchronize(s));
    *len = got[0] >= 0 ? got[0] : got[2];
    *sum = got[0] >= 0 ? got[1] : got[3];
    return MX_OK;
}

}  // namespace mxp

extern "C" int mx_select_device(int rows, int cols, int nnz, const int *rowPtr_dev, const int *colInd_dev, float tau_c,
                                float tau_r, int *descColId_dev, int *descRowId_dev, mx_selection *out, void *stream)
{
    static const char who[] = "mx_select_device";
    using namespace mxp;
    if (rows < 0 || cols < 0 || nnz < 0 || !rowPtr_dev || !out || (cols > 0 && !descColId_dev) ||
        (rows > 0 && !descRowId_dev) || (nnz > 0 && (!colInd_dev || rows == 0 || cols == 0)) || !(tau_c >= 0.f) ||
        !(tau_c <= 1.f) || !(tau_r >= 0.f) || !(tau_r <= tau_c)) {
        mx::set_error("mx_select_device: bad argument");
        return MX_ERR_ARG;
    }
    if (nnz > kMaxCount || rows > kMaxCount || cols > kMaxCount) {
        mx::set_error("mx_select_device: more than 2^31 - 513 entries, rows or columns");
        return MX_ERR_ARG;
    }
    hipStream_t s = (hipStream_t)stream;
    mx::MemScope scope(s);
    *out = mx_selection{0, 0, 0, 0};
    const size_t n = (size_t)std::max(rows, cols);
    size_t scanBytes = 0;
    if (n > 0) MXP_TRY(rocprim::inclusive_scan(nullptr, scanBytes, (const int *)nullptr, (int *)nullptr, n, rocprim::plus<int>(), s));
    const size_t digitB = (digit_bytes(n) + 255) & ~(size_t)255;
    // counts [n], work [3 n + 4], flag, dense flags [cols], the library's storage
    const size_t cntB = (n * sizeof(int) + 255) & ~(size_t)255, workB = ((3 * n + 4) * sizeof(int) + 255) & ~(size_t)255;
    const size_t denseB = ((size_t)cols + 255) & ~(size_t)255;
    Scratch scratch;
    MXP_TRY(mx::dev_malloc(&scratch.p, cntB + workB + 256 + denseB + digitB + scanBytes + 256));
    unsigned char *base = (unsigned char *)scratch.p;
    int *cnt = (int *)base, *work = (int *)(base + cntB), *bad = (int *)(base + cntB + workB);
    unsigned char *dense = base + cntB + workB + 256;
    int *digitTmp = (int *)(dense + denseB);
    void *scanTmp = dense + denseB + digitB;
    const int eblocks = (nnz + kBlock - 1) / kBlock;

    // ---- column pass (test/test_autotc_spmv.cpp:1122-1141)
    MXP_TRY(hipMemsetAsync(base, 0, cntB + workB + 256 + denseB, s));
    if (nnz >= kBucketCounts && mxd::buckets_hold(cols)) {
        const mxd::Buckets B = mxd::make_buckets(cols, nnz);
        const int tiles = (int)(((long long)nnz + mxd::kTile - 1) / mxd::kTile);
        const size_t countB = ((size_t)tiles * (B.n + 1) * 4 + 255) & ~(size_t)255, firstB = (2 * mxd::kDigits + 64) * sizeof(int);
        Scratch held;
        MXP_TRY(mx::dev_malloc(&held.p, countB + firstB + (size_t)nnz * 2));
        int *count = (int *)held.p, *badTile = count + (size_t)tiles * B.n, *first = (int *)((unsigned char *)held.p + countB), *total = first + mxd::kDigits + 1;
        unsigned short *column = (unsigned short *)((unsigned char *)held.p + countB + firstB);
        hipLaunchKernelGGL(mxd::bucket_counts_kernel, mxd::tile_blocks(tiles), dim3(mxd::kThreads), 0, s, colInd_dev, cols, nnz, B, tiles, count, badTile);
        hipLaunchKernelGGL(mxd::bucket_offsets_kernel, dim3((unsigned)((B.n + 15) / 16)), dim3(1024), 0, s, count, B.n, tiles, total);
        hipLaunchKernelGGL(mxd::bucket_starts_kernel<false>, dim3(1), dim3(mxd::kThreads), 0, s, (const int *)total, B.n, mxd::BucketBound{}, (const int *)badTile, tiles, first, bad);
        hipLaunchKernelGGL(bucket_columns_kernel, mxd::tile_blocks(tiles), dim3(mxd::kThreads), 0, s, colInd_dev, nnz, cols, B, tiles, (const int *)count,
                           (const int *)first, column);
        hipLaunchKernelGGL(count_columns_kernel, dim3((unsigned)B.n), dim3(mxd::kThreads), 0, s, (const unsigned short *)column, (const int *)first, cols, B, cnt);
        MXP_TRY(hipGetLastError());
    } else if (nnz > 0) {
        hipLaunchKernelGGL(index_histogram_kernel, dim3(eblocks), dim3(kBlock), 0, s, colInd_dev, nnz, cols, cnt, bad);
        MXP_TRY(hipGetLastError());
    }
    // (what the orders need to know of their counts comes down with the flag; a row has no more entries in selected columns than it has)
    if (n > 0)
        hipLaunchKernelGGL(highest_kernel, dim3((unsigned)std::min<size_t>(256, (n + kBlock - 1) / kBlock)), dim3(kBlock), 0, s, (const int *)cnt, cols, rowPtr_dev,
                           rows, bad + 1);
    MXP_TRY(hipGetLastError());
    int got[3] = {0, 0, 0};
    MXP_TRY(hipMemcpyAsync(got, bad, sizeof(got), hipMemcpyDeviceToHost, s));
    MXP_TRY(hipStreamSynchronize(s));
    if (got[0]) {
        mx::set_error("mx_select_device: column index out of range");
        return MX_ERR_ARG;
    }
    int rc = order_and_reach(cnt, cols, got[1], mx::threshold(nnz, tau_c), descColId_dev, work, digitTmp, scanTmp, scanBytes,
                             s, &out->dCols, &out->nnzColD);
    if (rc != MX_OK) return rc;

    // ---- row pass on the selected columns (:1240-1267)
    MXP_TRY(hipMemsetAsync(cnt, 0, cntB, s));
    if (out->dCols > 0) {
        hipLaunchKernelGGL(mark_selected_kernel, dim3((out->dCols + kBlock - 1) / kBlock), dim3(kBlock), 0, s,
                           (const int *)descColId_dev, out->dCols, dense);
        MXP_TRY(hipGetLastError());
    }
    if (nnz > 0) {
        hipLaunchKernelGGL(dense_row_counts_kernel, mxr::tile_grid(nnz), dim3(kBlock), 0, s, rowPtr_dev, colInd_dev,
                           (const unsigned char *)dense, rows, nnz, cnt);
        MXP_TRY(hipGetLastError());
    }
    rc = order_and_reach(cnt, rows, got[2], mx::threshold(nnz, tau_r), descRowId_dev, work, digitTmp, scanTmp, scanBytes, s,
                         &out->dRows, &out->nnzRowD);
    return rc;
}


extern "C" int mx_split_device(mx_dtype dtype, int rows, int cols, int nnz, const int *rowPtr_dev, const int *colInd_dev,
                               const void *val_dev, const mx_selection *sel, const int *descColId_dev,
                               const int *descRowId_dev, int *ddRowPtr_dev, int *ddColInd_dev, void *ddVal_dev,
                               int *cdRowPtr_dev, int *cdColInd_dev, void *cdVal_dev, void *stream)
{
    static const char who[] = "mx_split_device";
    using namespace mxp;
    if ((dtype != MX_F64 && dtype != MX_F16) || rows < 0 || cols < 0 || nnz < 0 || !sel || !rowPtr_dev || !ddRowPtr_dev ||
        !cdRowPtr_dev || sel->dCols < 0 || sel->dCols > cols || sel->dRows < 0 || sel->dRows > rows || sel->nnzRowD < 0 ||
        sel->nnzRowD > nnz || (sel->dCols > 0 && !descColId_dev) || (sel->dRows > 0 && !descRowId_dev) ||
        (nnz > 0 && (!colInd_dev || !val_dev || rows == 0 || cols == 0)) || (sel->nnzRowD > 0 && (!ddColInd_dev || !ddVal_dev)) ||
        (nnz - sel->nnzRowD > 0 && (!cdColInd_dev || !cdVal_dev))) {
        mx::set_error("mx_split_device: bad argument");
        return MX_ERR_ARG;
    }
    if (nnz > kMaxCount || rows > kMaxCount || cols > kMaxCount) {
        mx::set_error("mx_split_device: more than 2^31 - 513 entries, rows or columns");
        return MX_ERR_ARG;
    }
    hipStream_t s = (hipStream_t)stream;
    mx::MemScope scope(s);
    const int dCols = sel->dCols, dRows = sel->dRows, nDD = sel->nnzRowD;
    int colBits = 1, rowBits = 1;
    while (colBits < 31 && (1ll << colBits) < (long long)cols) ++colBits;
    while (rowBits < 31 && (1ll << rowBits) < (long long)rows) ++rowBits;
    const unsigned keyBits = (unsigned)(colBits + rowBits + 2);
    const size_t nScan = (size_t)std::max(rows, cols) + 1;
    size_t scanBytes = 0;
    MXP_TRY(rocprim::exclusive_scan(nullptr, scanBytes, (const int *)nullptr, (int *)nullptr, 0, nScan, rocprim::plus<int>(), s));
    auto al = [](size_t b) { return (b + 255) & ~(size_t)255; };
    const size_t colB = al(((size_t)cols + 1) * sizeof(int)), rowB = al(((size_t)rows + 1) * sizeof(int));
    const size_t denseB = al((size_t)cols + 1), listB = al(mxs::list_ints(nnz) * sizeof(int));
    // newCol, notSel, pos [cols+1]; rowRank, rcnt, cdLen, ddLen [rows+1]; dense; the lists of long rows
    Scratch scratch;
    MXP_TRY(mx::dev_malloc(&scratch.p, 3 * colB + 4 * rowB + denseB + listB + scanBytes + 512));
    unsigned char *b = (unsigned char *)scratch.p;
    int *newCol = (int *)b, *notSel = (int *)(b + colB), *pos = (int *)(b + 2 * colB);
    b += 3 * colB;
    int *rowRank = (int *)b, *rcnt = (int *)(b + rowB), *cdLen = (int *)(b + 2 * rowB), *ddLen = (int *)(b + 3 * rowB);
    b += 4 * rowB;
    unsigned char *dense = b;
    b += denseB;
    int *list = (int *)b;
    b += listB;
    void *scanTmp = b;
    int *bad = (int *)(b + al(scanBytes)), *classCount = bad + 1;  // in the spare bytes at the end
    auto grid = [](long long n) { return dim3((unsigned)((n + kBlock - 1) / kBlock)); };

    // the caller's arrays become addresses below: row pointers, column ids and both orders are
    // looked at first (1 = rowPtr, 2 = colInd, 4 = descColId, 8 = descRowId)
    MXP_TRY(hipMemsetAsync(bad, 0, (2 + mxs::kClasses) * sizeof(int), s));
    hipLaunchKernelGGL(pointer_check_kernel, grid((long long)rows + 1), dim3(kBlock), 0, s, rowPtr_dev, rows, nnz, 1, bad);
    if (nnz > 0) hipLaunchKernelGGL(range_check_kernel, grid(nnz), dim3(kBlock), 0, s, colInd_dev, nnz, cols, 2, bad);
    if (dCols > 0) hipLaunchKernelGGL(range_check_kernel, grid(dCols), dim3(kBlock), 0, s, descColId_dev, dCols, cols, 4, bad);
    if (dRows > 0) hipLaunchKernelGGL(range_check_kernel, grid(dRows), dim3(kBlock), 0, s, descRowId_dev, dRows, rows, 8, bad);
    MXP_TRY(hipGetLastError());
    MXP_TRY(mxs::classify_rows(rowPtr_dev, rows, nnz, list, classCount, s));
    mxs::RowClasses classes{};
    {
        int got[2 + mxs::kClasses] = {};
        MXP_TRY(hipMemcpyAsync(got, bad, sizeof(got), hipMemcpyDeviceToHost, s));
        MXP_TRY(hipStreamSynchronize(s));
        const int badHost = got[0];
        std::copy(got + 1, got + 2 + mxs::kClasses, classes.n);
        if (badHost) {
            mx::set_error(std::string("mx_split_device: ") + ((badHost & 1) ? "rowPtr does not rise from 0 to nnz" :
                          (badHost & 2) ? "column index out of range" : (badHost & 4) ? "descColId entry out of range" :
                          "descRowId entry out of range"));
            return MX_ERR_ARG;
        }
    }

    // new column ids: rank for a selected column, dCols + position among the others otherwise
    MXP_TRY(hipMemsetAsync(dense, 0, denseB, s));
    MXP_TRY(hipMemsetAsync(rowRank, 0xff, rowB, s));  // -1
    MXP_TRY(hipMemsetAsync(rcnt, 0, rowB, s));
    if (dCols > 0) {
        hipLaunchKernelGGL(mark_selected_kernel, grid(dCols), dim3(kBlock), 0, s, descColId_dev, dCols, dense);
        hipLaunchKernelGGL(scatter_rank_kernel, grid(dCols), dim3(kBlock), 0, s, descColId_dev, dCols, newCol);
    }
    hipLaunchKernelGGL(not_selected_kernel, grid((long long)cols + 1), dim3(kBlock), 0, s, (const unsigned char *)dense, cols, notSel);
    MXP_TRY(hipGetLastError());
    MXP_TRY(rocprim::exclusive_scan(scanTmp, scanBytes, (const int *)notSel, pos, 0, (size_t)cols + 1, rocprim::plus<int>(), s));
    if (cols > 0)
        hipLaunchKernelGGL(sparse_columns_kernel, grid(cols), dim3(kBlock), 0, s, (const unsigned char *)dense, (const int *)pos, cols,
                           dCols, newCol);
    // rows: rank of the selected ones, counts inside the selected columns, lengths, pointers
    if (dRows > 0) hipLaunchKernelGGL(scatter_rank_kernel, grid(dRows), dim3(kBlock), 0, s, descRowId_dev, dRows, rowRank);
    if (nnz > 0)
        hipLaunchKernelGGL(dense_row_counts_kernel, mxr::tile_grid(nnz), dim3(kBlock), 0, s, rowPtr_dev, colInd_dev,
                           (const unsigned char *)dense, rows, nnz, rcnt);
    hipLaunchKernelGGL(split_lengths_kernel, grid((long long)rows + 1), dim3(kBlock), 0, s, rowPtr_dev, (const int *)rcnt,
                       (const int *)rowRank, descRowId_dev, rows, dRows, cdLen, ddLen);
    MXP_TRY(hipGetLastError());
    MXP_TRY(rocprim::exclusive_scan(scanTmp, scanBytes, (const int *)cdLen, cdRowPtr_dev, 0, (size_t)rows + 1, rocprim::plus<int>(), s));
    MXP_TRY(rocprim::exclusive_scan(scanTmp, scanBytes, (const int *)ddLen, ddRowPtr_dev, 0, (size_t)dRows + 1, rocprim::plus<int>(), s));
    // the totals must be what the caller sized the outputs for
    int totals[2] = {0, 0};
    MXP_TRY(hipMemcpyAsync(&totals[0], ddRowPtr_dev + dRows, sizeof(int), hipMemcpyDeviceToHost, s));
    MXP_TRY(hipMemcpyAsync(&totals[1], cdRowPtr_dev + rows, sizeof(int), hipMemcpyDeviceToHost, s));
    MXP_TRY(hipStreamSynchronize(s));
    if (totals[0] != nDD || totals[1] != nnz - nDD) {
        mx::set_error("mx_split_device: the selection does not belong to this matrix (entry totals differ)");
        return MX_ERR_ARG;
    }
    if (nnz > 0 && classes.n[mxs::kClasses] == 0) {
        auto split = [&](auto *ddVal, auto *cdVal, auto *val) -> hipError_t {
            typedef typename std::remove_pointer<decltype(ddVal)>::type V;
            const SplitRows<V> io{rowPtr_dev, colInd_dev, newCol, rowRank, rcnt, ddRowPtr_dev, cdRowPtr_dev, val, dCols, colBits,
                                  ddColInd_dev, ddVal, cdColInd_dev, cdVal};
            return mxs::sort_rows(rowPtr_dev, rows, nnz, list, classes, io, s);
        };
        if (dtype == MX_F64) MXP_TRY(split((double *)ddVal_dev, (double *)cdVal_dev, (const double *)val_dev));
        else MXP_TRY(split((uint16_t *)ddVal_dev, (uint16_t *)cdVal_dev, (const uint16_t *)val_dev));
    } else if (nnz > 0) {
        size_t sortBytes = 0;
        MXP_TRY(rocprim::radix_sort_pairs(nullptr, sortBytes, (const unsigned long long *)nullptr, (unsigned long long *)nullptr,
                                          (const int *)nullptr, (int *)nullptr, (size_t)nnz, 0u, keyBits, s));
        const size_t keyB = al((size_t)nnz * 8), payB = al((size_t)nnz * 4);
        Scratch sort;
        MXP_TRY(mx::dev_malloc(&sort.p, 2 * keyB + 2 * payB + sortBytes + 256));
        b = (unsigned char *)sort.p;
        unsigned long long *keyIn = (unsigned long long *)b, *keyOut = (unsigned long long *)(b + keyB);
        int *payIn = (int *)(b + 2 * keyB), *payOut = (int *)(b + 2 * keyB + payB);
        void *sortTmp = b + 2 * keyB + 2 * payB;
        hipLaunchKernelGGL(split_keys_kernel, mxr::tile_grid(nnz), dim3(kBlock), 0, s, rowPtr_dev, colInd_dev, (const int *)newCol,
                           (const int *)rowRank, rows, nnz, dCols, colBits, rowBits, keyIn, payIn);
        MXP_TRY(hipGetLastError());
        MXP_TRY(rocprim::radix_sort_pairs(sortTmp, sortBytes, (const unsigned long long *)keyIn, keyOut, (const int *)payIn, payOut,
                                          (size_t)nnz, 0u, keyBits, s));
        if (dtype == MX_F64)
            hipLaunchKernelGGL(split_gather_kernel<double>, grid(nnz), dim3(kBlock), 0, s, (const unsigned long long *)keyOut,
                               (const int *)payOut, (const double *)val_dev, nnz, nDD, colBits, ddColInd_dev, (double *)ddVal_dev,
                               cdColInd_dev, (double *)cdVal_dev);
        else
            hipLaunchKernelGGL(split_gather_kernel<uint16_t>, grid(nnz), dim3(kBlock), 0, s, (const unsigned long long *)keyOut,
                               (const int *)payOut, (const uint16_t *)val_dev, nnz, nDD, colBits, ddColInd_dev,
                               (uint16_t *)ddVal_dev, cdColInd_dev, (uint16_t *)cdVal_dev);
        MXP_TRY(hipGetLastError());
    }
    return MX_OK;  // (the scope waits for the stream before it hands the scratch on)
}


extern "C" void mx_tiles_device_free(mx_device_tiles *t)
{
    if (!t) return;
    if (t->base) (void)mx::dev_free(t->base);
    *t = mx_device_tiles{};
}

extern "C" int mx_tiles_device(mx_dtype dtype, int dRows, int dCols, int nnzRowD, const int *ddRowPtr_dev,
                               const int *ddColInd_dev, const void *ddVal_dev, mx_device_tiles *out, void *stream)
{
    static const char who[] = "mx_tiles_device";
    using namespace mxp;
    if ((dtype != MX_F64 && dtype != MX_F16) || dRows < 0 || dCols < 0 || nnzRowD < 0 || !out || !ddRowPtr_dev ||
        (nnzRowD > 0 && (!ddColInd_dev || !ddVal_dev || dRows == 0 || dCols == 0))) {
        mx::set_error("mx_tiles_device: bad argument");
        return MX_ERR_ARG;
    }
    if (nnzRowD > kMaxCount || dRows > kMaxCount || dCols > kMaxCount) {
        mx::set_error("mx_tiles_device: more than 2^31 - 513 entries, rows or columns");
        return MX_ERR_ARG;
    }
    hipStream_t s = (hipStream_t)stream;
    mx::MemScope scope(s);
    *out = mx_device_tiles{};
    const int fragK = mx::frag_k(dtype), n = nnzRowD, chunkNum = (dRows + mx::kFragM - 1) / mx::kFragM;
    const size_t es = (size_t)mx::elem_size(dtype);
    int colBits = 1, chunkBits = 1;
    while (colBits < 31 && (1ll << colBits) < (long long)dCols) ++colBits;
    // (chunkBits: of the numbers of the chunks that the radix sort is for; all keys are shifted by colBits alone)
    auto al = [](size_t b) { return (b + 255) & ~(size_t)255; };
    auto grid = [](long long m) { return dim3((unsigned)((m + kBlock - 1) / kBlock)); };
    size_t scanBytes = 0;
    MXP_TRY(rocprim::inclusive_scan(nullptr, scanBytes, (const int *)nullptr, (int *)nullptr,
                                    (size_t)std::max(n, chunkNum) + 1, rocprim::plus<int>(), s));
    {   // the exclusive form may ask for a different amount: take the larger
        size_t b2 = 0;
        MXP_TRY(rocprim::exclusive_scan(nullptr, b2, (const int *)nullptr, (int *)nullptr, 0, (size_t)std::max(n, chunkNum) + 1,
                                        rocprim::plus<int>(), s));
        scanBytes = std::max(scanBytes, b2);
    }
    scanBytes = al(scanBytes);
    // scratch: sorted keys and payloads, heads, their running count, ecr, per-chunk fragments and first entries, lists
    const size_t keyB = al((size_t)n * 8), intB = al(((size_t)n + 1) * 4), chB = al(((size_t)chunkNum + 1) * 4);
    const size_t listB = al(mxs::list_ints(n) * 4);
    Scratch scratch;
    MXP_TRY(mx::dev_malloc(&scratch.p, keyB + 4 * intB + 3 * chB + listB + scanBytes + 256));
    unsigned char *b = (unsigned char *)scratch.p;
    unsigned long long *keyOut = (unsigned long long *)b;
    b += keyB;
    int *payOut = (int *)b, *head = (int *)(b + intB), *run = (int *)(b + 2 * intB), *ecr = (int *)(b + 3 * intB);
    b += 4 * intB;
    int *frags = (int *)b, *chunkPtrTmp = (int *)(b + chB), *chunkFirst = (int *)(b + 2 * chB);
    b += 3 * chB;
    int *list = (int *)b;
    b += listB;
    void *scanTmp = b;
    mxs::RowClasses classes{};
    int nLong = 0;  // entries up to the end of the last chunk that a workgroup has no room for
    {
        // the caller's A_dd is about to be used for addressing: pointers and column ids are looked at first
        int *bad = (int *)((unsigned char *)scanTmp + scanBytes);  // in the 256 spare bytes at the end
        MXP_TRY(hipMemsetAsync(bad, 0, (4 + mxs::kClasses) * sizeof(int), s));
        hipLaunchKernelGGL(pointer_check_kernel, grid((long long)dRows + 1), dim3(kBlock), 0, s, ddRowPtr_dev, dRows, n, 1, bad);
        if (n > 0) hipLaunchKernelGGL(range_check_kernel, grid(n), dim3(kBlock), 0, s, ddColInd_dev, n, dCols, 2, bad);
        hipLaunchKernelGGL(chunk_starts_kernel, grid((long long)chunkNum + 1), dim3(kBlock), 0, s, ddRowPtr_dev, dRows, chunkNum, chunkFirst);
        hipLaunchKernelGGL(long_chunks_kernel, grid((long long)chunkNum + 1), dim3(kBlock), 0, s, (const int *)chunkFirst, chunkNum, bad + 1,
                           bad + 3 + mxs::kClasses);
        MXP_TRY(hipGetLastError());
        MXP_TRY(mxs::classify_rows(chunkFirst, chunkNum, n, list, bad + 2, s));
        int got[4 + mxs::kClasses] = {};
        MXP_TRY(hipMemcpyAsync(got, bad, sizeof(got), hipMemcpyDeviceToHost, s));
        MXP_TRY(hipStreamSynchronize(s));
        const int badHost = got[0];
        nLong = got[1];
        while (chunkBits < 31 && (1ll << chunkBits) < (long long)got[3 + mxs::kClasses]) ++chunkBits;
        std::copy(got + 2, got + 3 + mxs::kClasses, classes.n);
        if (badHost) {
            mx::set_error((badHost & 1) ? "mx_tiles_device: ddRowPtr does not rise from 0 to nnzRowD"
                                        : "mx_tiles_device: column index out of range");
            return MX_ERR_ARG;
        }
    }

    // distinct columns per chunk: sort by (chunk, column), mark first occurrences, count them
    if (n > 0) {
        MXP_TRY(mxs::sort_rows(chunkFirst, chunkNum, n, list, classes, ChunkColumns{ddColInd_dev, colBits, keyOut, payOut}, s));
        if (nLong > 0) {
            size_t sortBytes = 0;
            MXP_TRY(rocprim::radix_sort_pairs(nullptr, sortBytes, (const unsigned long long *)nullptr, (unsigned long long *)nullptr,
                                              (const int *)nullptr, (int *)nullptr, (size_t)nLong, 0u, (unsigned)(colBits + chunkBits), s));
            Scratch sort;
            const size_t inB = al((size_t)nLong * 8), payB = al((size_t)nLong * 4);
            MXP_TRY(mx::dev_malloc(&sort.p, inB + payB + sortBytes + 256));
            unsigned long long *keyIn = (unsigned long long *)sort.p;
            int *payIn = (int *)((unsigned char *)sort.p + inB);
            hipLaunchKernelGGL(tile_keys_kernel, mxr::tile_grid(nLong), dim3(kBlock), 0, s, (const int *)chunkFirst, ddColInd_dev, chunkNum, nLong,
                               colBits, keyIn, payIn);
            MXP_TRY(hipGetLastError());
            MXP_TRY(rocprim::radix_sort_pairs((unsigned char *)sort.p + inB + payB, sortBytes, (const unsigned long long *)keyIn, keyOut,
                                              (const int *)payIn, payOut, (size_t)nLong, 0u, (unsigned)(colBits + chunkBits), s));
        }
        hipLaunchKernelGGL(tile_heads_kernel, grid(n), dim3(kBlock), 0, s, (const unsigned long long *)keyOut, n, head);
        MXP_TRY(hipGetLastError());
        MXP_TRY(rocprim::inclusive_scan(scanTmp, scanBytes, (const int *)head, run, (size_t)n, rocprim::plus<int>(), s));
    }
    hipLaunchKernelGGL(tile_chunk_frags_kernel, grid((long long)chunkNum + 1), dim3(kBlock), 0, s, ddRowPtr_dev, (const int *)run,
                       dRows, chunkNum, fragK, frags);
    MXP_TRY(hipGetLastError());
    // chunkPtr lives in the output block, whose size needs the total first
    MXP_TRY(rocprim::exclusive_scan(scanTmp, scanBytes, (const int *)frags, chunkPtrTmp, 0, (size_t)chunkNum + 1, rocprim::plus<int>(), s));
    int totalTcFrags = 0;
    MXP_TRY(hipMemcpyAsync(&totalTcFrags, chunkPtrTmp + chunkNum, sizeof(int), hipMemcpyDeviceToHost, s));
    MXP_TRY(hipStreamSynchronize(s));

    // output block: chunkPtr, sparse_AToX_index, fragPtr, fragBit (64-bit while it is built), tcVal (at most n)
    const size_t cpB = al(((size_t)chunkNum + 1) * 4), axB = al((size_t)totalTcFrags * fragK * 4 + 4),
                 fpB = al(((size_t)totalTcFrags + 1) * 4), fbB = al((size_t)totalTcFrags * 8 + 8), tvB = al((size_t)n * es + 8);
    Scratch outBlock;
    MXP_TRY(mx::dev_malloc(&outBlock.p, cpB + axB + fpB + fbB + tvB));
    unsigned char *o = (unsigned char *)outBlock.p;
    int *chunkPtr = (int *)o, *atox = (int *)(o + cpB), *fragPtr = (int *)(o + cpB + axB);
    unsigned long long *bits = (unsigned long long *)(o + cpB + axB + fpB);
    void *tcVal = o + cpB + axB + fpB + fbB;
    MXP_TRY(hipMemcpyAsync(chunkPtr, chunkPtrTmp, ((size_t)chunkNum + 1) * 4, hipMemcpyDeviceToDevice, s));
    MXP_TRY(hipMemsetAsync(atox, 0, axB + fpB + fbB, s));  // padding of the column lists is zero (:1380-1404)
    if (n > 0) {
        hipLaunchKernelGGL(tile_rank_kernel, grid(n), dim3(kBlock), 0, s, (const unsigned long long *)keyOut, (const int *)payOut,
                           (const int *)head, (const int *)run, ddRowPtr_dev, (const int *)chunkPtr, dRows, n, colBits, fragK, ecr,
                           atox, bits);
        MXP_TRY(hipGetLastError());
    }
    // fragPtr: running count of the set bits.  head[] is free again and long enough only when
    // totalTcFrags <= n, which holds (every fragment has an entry) -- but take no chances:
    if (totalTcFrags > n) {
        mx::set_error("mx_tiles_device: more fragments than entries (ddRowPtr is not A_dd's)");
        return MX_ERR_ARG;
    }
    hipLaunchKernelGGL(tile_popcount_kernel, grid((long long)totalTcFrags + 1), dim3(kBlock), 0, s, (const unsigned long long *)bits,
                       totalTcFrags, head);
    MXP_TRY(hipGetLastError());
    MXP_TRY(rocprim::exclusive_scan(scanTmp, scanBytes, (const int *)head, fragPtr, 0, (size_t)totalTcFrags + 1, rocprim::plus<int>(), s));
    if (n > 0) {
        if (dtype == MX_F64)
            hipLaunchKernelGGL(tile_values_kernel<double>, mxr::tile_grid(n), dim3(kBlock), 0, s, ddRowPtr_dev, ddColInd_dev,
                               (const double *)ddVal_dev, (const int *)ecr, (const int *)chunkPtr, (const int *)fragPtr,
                               (const unsigned long long *)bits, dRows, n, fragK, (double *)tcVal);
        else
            hipLaunchKernelGGL(tile_values_kernel<uint16_t>, mxr::tile_grid(n), dim3(kBlock), 0, s, ddRowPtr_dev, ddColInd_dev,
                               (const uint16_t *)ddVal_dev, (const int *)ecr, (const int *)chunkPtr, (const int *)fragPtr,
                               (const unsigned long long *)bits, dRows, n, fragK, (uint16_t *)tcVal);
        MXP_TRY(hipGetLastError());
    }
    if (dtype == MX_F64 && totalTcFrags > 0) {  // 8 x 4 bits: the reference keeps them in 32-bit words
        // narrowed in place, front to back: word f of the narrow form lies below word f of the wide one,
        // but another thread may still need it -- go through the free scratch instead
        hipLaunchKernelGGL(narrow_bits_kernel, grid(totalTcFrags), dim3(kBlock), 0, s, (const unsigned long long *)bits, totalTcFrags,
                           (unsigned *)run);
        MXP_TRY(hipGetLastError());
        MXP_TRY(hipMemcpyAsync(bits, run, (size_t)totalTcFrags * 4, hipMemcpyDeviceToDevice, s));
    }
    int tcValCount = 0;
    MXP_TRY(hipMemcpyAsync(&tcValCount, fragPtr + totalTcFrags, sizeof(int), hipMemcpyDeviceToHost, s));
    MXP_TRY(hipStreamSynchronize(s));
    out->chunkNum = chunkNum;
    out->totalTcFrags = totalTcFrags;
    out->fragK = fragK;
    out->tcValCount = tcValCount;
    out->chunkPtr = chunkPtr;
    out->sparse_AToX_index = atox;
    out->fragPtr = fragPtr;
    out->fragBit = bits;
    out->tcVal = tcVal;
    out->base = outBlock.p;
    outBlock.p = nullptr;  // the caller's now
    return MX_OK;
}


// mx_partition_create with the extraction done on the device: the matrix is uploaded, selected,
// split and encoded there (mx_select_device, mx_split_device, mx_tiles_device) and the arrays come
// back into the same host structure, so that everything downstream (plans, files, the checksum)
// cannot tell the two routes apart.
// The device arrays of a partition made here (mx_partition::twin) and their way down.
namespace {
void twin_free(void *w)
{
    mx::PartitionTwin *W = (mx::PartitionTwin *)w;
    if (!W) return;
    mx::IdleFrees idle;
    (void)mx::dev_free(W->order);
    (void)mx::dev_free(W->split);
    mx_tiles_device_free(&W->T);
    delete W;
}
// fills the host vectors of P from its twin
int twin_download(mx_partition *P)
{
    using namespace mxp;
    static const char who[] = "mx_partition_create_device (arrays to the host)";
    const mx::PartitionTwin &W = *(const mx::PartitionTwin *)P->twin;
    const int rows = W.rows, cols = W.cols, nDD = W.nDD, nCD = W.nCD, dRows = W.dRows, dCols = W.dCols;
    const size_t es = (size_t)mx::elem_size(W.dtype);
    const mx_device_tiles &T = W.T;
    try {
        P->descColId.resize(cols);
        P->rId.resize(dRows);
        P->ddRowPtr.resize((size_t)dRows + 1);
        P->ddColInd.resize(nDD);
        P->ddVal.resize(nDD, (int)es);
        P->cdRowPtr.resize((size_t)rows + 1);
        P->cdColInd.resize(nCD);
        P->cdVal.resize(nCD, (int)es);
        P->chunkPtr.resize((size_t)T.chunkNum + 1);
        P->sparse_AToX_index.resize((size_t)T.totalTcFrags * T.fragK);
        P->fragPtr.resize((size_t)T.totalTcFrags + 1);
        if (W.dtype == MX_F64) P->fragBit32.resize(T.totalTcFrags);
        else P->fragBit64.resize(T.totalTcFrags);
        P->tcVal.resize(T.tcValCount, (int)es);
    } catch (const std::bad_alloc &) {
        mx::set_error("mx_partition_create_device: out of memory");
        return MX_ERR_ALLOC;
    }
    auto down = [](void *dst, const void *src, size_t bytes) {
        return bytes ? hipMemcpy(dst, src, bytes, hipMemcpyDeviceToHost) : hipSuccess;
    };
    MXP_TRY(down(P->descColId.data(), W.dc, (size_t)cols * 4));
    MXP_TRY(down(P->rId.data(), W.dr, (size_t)dRows * 4));
    MXP_TRY(down(P->ddRowPtr.data(), W.ddp, ((size_t)dRows + 1) * 4));
    MXP_TRY(down(P->ddColInd.data(), W.ddc, (size_t)nDD * 4));
    MXP_TRY(down(P->ddVal.data(), W.ddv, (size_t)nDD * es));
    MXP_TRY(down(P->cdRowPtr.data(), W.cdp, ((size_t)rows + 1) * 4));
    MXP_TRY(down(P->cdColInd.data(), W.cdc, (size_t)nCD * 4));
    MXP_TRY(down(P->cdVal.data(), W.cdv, (size_t)nCD * es));
    MXP_TRY(down(P->chunkPtr.data(), T.chunkPtr, ((size_t)T.chunkNum + 1) * 4));
    MXP_TRY(down(P->sparse_AToX_index.data(), T.sparse_AToX_index, (size_t)T.totalTcFrags * T.fragK * 4));
    MXP_TRY(down(P->fragPtr.data(), T.fragPtr, ((size_t)T.totalTcFrags + 1) * 4));
    if (W.dtype == MX_F64) MXP_TRY(down(P->fragBit32.data(), T.fragBit, (size_t)T.totalTcFrags * 4));
    else MXP_TRY(down(P->fragBit64.data(), T.fragBit, (size_t)T.totalTcFrags * 8));
    MXP_TRY(down(P->tcVal.data(), T.tcVal, (size_t)T.tcValCount * es));
    // the lists of what was not selected, ascending (test/test_autotc_spmv.cpp:1143-1160, :1261-1277)
    std::vector<unsigned char> taken((size_t)std::max(rows, cols), 0);
    for (int i = 0; i < dCols; ++i) taken[P->descColId[i]] = 1;
    P->newArray.clear();
    P->newArray.reserve(P->sCols);
    for (int c = 0; c < cols; ++c)
        if (!taken[c]) P->newArray.push_back(c);
    std::fill(taken.begin(), taken.end(), 0);
    for (int i = 0; i < dRows; ++i) taken[P->rId[i]] = 1;
    P->newArray_.clear();
    P->newArray_.reserve(P->sRows);
    for (int r = 0; r < rows; ++r)
        if (!taken[r]) P->newArray_.push_back(r);
    P->host_ready = true;
    return MX_OK;
}
}  // namespace

extern "C" int mx_partition_create_device(const mx_csr *A, float tau_c, float tau_r, mx_partition **out)
{
    static const char who[] = "mx_partition_create_device";
    using namespace mxp;
    const int ok = mx::check_partition_args(A, tau_c, tau_r, out);
    if (ok != MX_OK) return ok;
    if (tau_c == 0.0f && tau_r == 0.0f) return mx_partition_create(A, tau_c, tau_r, out);  // nothing to extract
    int ndev = 0;
    if (hipGetDeviceCount(&ndev) != hipSuccess || ndev < 1) {
        mx::set_error("mx_partition_create_device: no HIP device");
        return MX_ERR_DEVICE;
    }
    (void)who;
    mx::MemScope scope(nullptr);
    const int rows = A->rows, cols = A->cols, nnz = A->nnz;
    const size_t es = (size_t)mx::elem_size(A->dtype);
    auto al = [](size_t b) { return (b + 255) & ~(size_t)255; };
    mx::PartitionTwin *W = new (std::nothrow) mx::PartitionTwin();
    if (!W) {
        mx::set_error("mx_partition_create_device: out of memory");
        return MX_ERR_ALLOC;
    }
    struct TwinGuard {
        mx::PartitionTwin *w;
        ~TwinGuard() { twin_free(w); }
    } wg{W};
    W->dtype = A->dtype;
    W->rows = rows;
    W->cols = cols;
    W->nnz = nnz;
    // the matrix (released when the extraction is done) and the two orders (kept)
    const size_t rpB = al(((size_t)rows + 1) * 4), ciB = al((size_t)nnz * 4 + 4), vaB = al((size_t)nnz * es + 8),
                 dcB = al((size_t)cols * 4 + 4), drB = al((size_t)rows * 4 + 4);
    Scratch in;
    MXP_TRY(mx::dev_malloc(&in.p, rpB + ciB + vaB));
    unsigned char *b = (unsigned char *)in.p;
    int *rp = (int *)b, *ci = (int *)(b + rpB);
    void *va = b + rpB + ciB;
    MXP_TRY(mx::dev_malloc(&W->order, dcB + drB));
    W->dc = (int *)W->order;
    W->dr = (int *)((unsigned char *)W->order + dcB);
    int *dc = W->dc, *dr = W->dr;
    MXP_TRY(mx::copy_up(rp, A->rowPtr, ((size_t)rows + 1) * 4));
    if (nnz > 0) {
        MXP_TRY(mx::copy_up(ci, A->colInd, (size_t)nnz * 4));
        MXP_TRY(mx::copy_up(va, A->val, (size_t)nnz * es));
    }
    mx_selection sel{};
    int rc = mx_select_device(rows, cols, nnz, rp, ci, tau_c, tau_r, dc, dr, &sel, nullptr);
    if (rc != MX_OK) return rc;
    const int nDD = sel.nnzRowD, nCD = nnz - nDD;
    const size_t ddpB = al(((size_t)sel.dRows + 1) * 4), ddcB = al((size_t)nDD * 4 + 4), ddvB = al((size_t)nDD * es + 8),
                 cdpB = al(((size_t)rows + 1) * 4), cdcB = al((size_t)nCD * 4 + 4), cdvB = al((size_t)nCD * es + 8);
    MXP_TRY(mx::dev_malloc(&W->split, ddpB + ddcB + ddvB + cdpB + cdcB + cdvB));
    b = (unsigned char *)W->split;
    W->ddp = (int *)b;
    W->ddc = (int *)(b + ddpB);
    W->ddv = b + ddpB + ddcB;
    W->cdp = (int *)(b + ddpB + ddcB + ddvB);
    W->cdc = (int *)(b + ddpB + ddcB + ddvB + cdpB);
    W->cdv = b + ddpB + ddcB + ddvB + cdpB + cdcB;
    rc = mx_split_device(A->dtype, rows, cols, nnz, rp, ci, va, &sel, dc, dr, W->ddp, W->ddc, W->ddv, W->cdp, W->cdc, W->cdv, nullptr);
    if (rc != MX_OK) return rc;
    rc = mx_tiles_device(A->dtype, sel.dRows, sel.dCols, nDD, W->ddp, W->ddc, W->ddv, &W->T, nullptr);
    if (rc != MX_OK) return rc;
    W->dRows = sel.dRows;
    W->dCols = sel.dCols;
    W->nDD = nDD;
    W->nCD = nCD;
    const mx_device_tiles &T = W->T;

    mx_partition *P = new (std::nothrow) mx_partition();
    if (!P) {
        mx::set_error("mx_partition_create_device: out of memory");
        return MX_ERR_ALLOC;
    }
    // the counts; the arrays stay on the device until somebody asks for them (mx::partition_host)
    P->dtype = A->dtype;
    P->rows = rows;
    P->cols = cols;
    P->nnz = nnz;
    P->fragM = mx::kFragM;
    P->fragK = mx::frag_k(A->dtype);
    P->tau_c = tau_c;
    P->tau_r = tau_r;
    P->extracted = true;
    P->dCols = sel.dCols;
    P->sCols = cols - sel.dCols;
    P->nnzColD = sel.nnzColD;
    P->nnzColS = nnz - sel.nnzColD;
    P->cols_ratio = (float)sel.dCols / (float)cols;
    P->dRows = sel.dRows;
    P->sRows = rows - sel.dRows;
    P->nnzRowD = nDD;
    P->nnzRowS = sel.nnzColD - nDD;
    P->nnzCD = nCD;
    P->chunkNum = T.chunkNum;
    P->totalTcFrags = T.totalTcFrags;
    P->tcValCount = T.tcValCount;
    P->tc_nnz_ratio = (double)nDD / ((double)T.totalTcFrags * mx::kFragM * P->fragK);
    P->host_ready = false;
    P->twin = W;
    P->twin_download = twin_download;
    P->twin_free = twin_free;
    wg.w = nullptr;  // the partition owns the twin now
    *out = P;
    return MX_OK;
}

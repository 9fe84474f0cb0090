// The slice layout of the CSR part (see DeviceSlices) built on the device from a CSR matrix that
// lives in device memory: the same arrays, byte for byte, as the host route (build_slices in
// mx_host_layout.cpp), for matrices that are already in HBM and for plans of large matrices, whose
// layout the host cores take a second to make.  The reference has no counterpart: its CSR
// kernel reads the CSR arrays as they are (src/spmv_kernel/cdSpMV.cu:407-418).
//
// What depends on every entry or every virtual row runs here: rows put in ascending column
// order (a stable sort by (row, column) when some row is not), virtual rows cut at slice borders
// and at the cap, their stable sort by (slice, length descending, kind of row), the entries
// placed into the lanes' streams, the lists the combine kernel walks.  What depends on chunks
// only (64 virtual rows each) -- which workgroup and wave streams which chunk -- is decided by
// plan_chunks_device (mx_chunks.hip) as plan_slice_chunks decides it on the host.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdint>
#include <cstring>
#include <string>
#include <vector>

#include <rocprim/device/device_radix_sort.hpp>
#include <rocprim/device/device_scan.hpp>

#include "mx_chunks.h"
#include "mx_device.h"
#include "mx_entry_rows.h"
#include "mx_internal.h"
#include "mx_row_sort.h"

namespace mxl {

// The order of a row's entries by column, made inside their workgroups.
struct RowColumns {
    const int *col;
    int *ord;
    __device__ __forceinline__ unsigned key(int, int e) const { return (unsigned)col[e]; }
    __device__ __forceinline__ void put(int, int, unsigned, int e, int k) const { ord[k] = e; }
};

__global__ __launch_bounds__(kBlock) void sort_keys_kernel(const int *__restrict__ rowPtr, const int *__restrict__ col, int rows, int nnz,
                                                           int colBits, unsigned long long *__restrict__ key, int *__restrict__ pay)
{
    __shared__ mxr::TileRows T;
    const int t0 = blockIdx.x * mxr::kTile;
    mxr::tile_rows(rowPtr, rows, nnz, t0, T);
#pragma unroll
    for (int j = 0; j < mxr::kPer; ++j) {
        const int i = j * kBlock + threadIdx.x, k = t0 + i;
        if (i >= nnz - t0) break;
        key[k] = ((unsigned long long)(unsigned)T.row[i] << colBits) | (unsigned)col[k];
        pay[k] = k;
    }
}

// ---- virtual rows ----
// Where the virtual rows start, a bit per entry (of a tile of kTile entries kWords words) and their number per tile.  A virtual
// row starts at every cap-th entry of a run, the entries of a row in one slice; the run that a tile begins in is searched for, the rest is
// found among the tile's own.  ord: the entries in ascending columns inside their rows, null where they are taken to lie so; then
// *flag |= 1 where they do not, and nothing else is to be used.
// (7.6 million entries in 700 thousand rows: rows and order of every entry, run heads, their running maximum, starts and their running sum,
// 200 us with the records, in arrays of the length of the matrix; so 68.)
constexpr int kWords = mxr::kTile / 64;
template <int SW>
__global__ __launch_bounds__(kBlock) void vrow_starts_kernel(const int *__restrict__ rowPtr, const int *__restrict__ col, const int *__restrict__ ord,
                                                             int rows, int nnz, int cap, unsigned long long *__restrict__ startBits,
                                                             int *__restrict__ tileStarts, int *__restrict__ flag)
{
    __shared__ mxr::TileRows T;
    __shared__ unsigned long long heads[kWords];
    __shared__ int carry, starts;
    const int t0 = blockIdx.x * mxr::kTile, tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
    mxr::tile_rows(rowPtr, rows, nnz, t0, T);
    auto column = [&](int k) { return col[ord ? ord[k] : k]; };
    if (w == 0) {
        // the first entry of the run that entry t0 belongs to: the row's first in a slice that is not before t0's
        const int q = column(t0) / SW;
        int lo = min(rowPtr[T.row[0]], t0), hi = t0;
        while (lo < hi) {
            const int step = (hi - lo + 63) / 64;
            const long long at = lo + (long long)lane * step;
            const int before = __popcll(__ballot(at < hi && column((int)min(at, (long long)t0)) / SW < q));
            if (before == 0) break;
            hi = (int)min((long long)hi, lo + (long long)before * step);
            lo += (before - 1) * step + 1;
        }
        if (lane == 0) {
            carry = lo;
            starts = 0;
        }
    }
    bool descends = false;
    int c[mxr::kPer];
#pragma unroll
    for (int j = 0; j < mxr::kPer; ++j) c[j] = column(t0 + min(j * kBlock + tid, nnz - 1 - t0));
#pragma unroll
    for (int j = 0; j < mxr::kPer; ++j) {
        const int i = j * kBlock + tid, k = t0 + i;
        int before = __shfl_up(c[j], 1);
        bool head = false;
        if (i < nnz - t0) {
            const int r = T.row[i];
            if (i > 0 ? T.row[i - 1] != r : rowPtr[r] == k) {
                head = true;
            } else {
                if (lane == 0) before = column(k - 1);
                head = before / SW != c[j] / SW;
                descends |= c[j] < before;
            }
        }
        const unsigned long long m = __ballot(head);
        if (lane == 0) heads[j * (kBlock / 64) + w] = m;
    }
    if (!ord && __any(descends) && lane == 0 && *(volatile int *)flag == 0) atomicOr(flag, 1);
    __syncthreads();
    int mine = 0;
#pragma unroll
    for (int j = 0; j < mxr::kPer; ++j) {
        const int i = j * kBlock + tid, k = t0 + i, word = j * (kBlock / 64) + w;
        // the last head at or before the entry: in its word, in an earlier one, or the carry
        const unsigned long long m = heads[word] & (~0ull >> (63 - lane));
        const unsigned long long some = __ballot(lane < word && heads[min(lane, kWords - 1)] != 0);
        int run = carry;
        if (m) run = t0 + word * 64 + 63 - __builtin_clzll(m);
        else if (some) {
            const int v = 63 - __builtin_clzll(some);
            run = t0 + v * 64 + 63 - __builtin_clzll(heads[v]);
        }
        const int d = k - run;  // (hardly any run is longer than cap: the division is for waves that have one)
        const unsigned long long s = __ballot(i < nnz - t0 && (d == 0 || (d >= cap && d % cap == 0)));
        if (lane == 0 && t0 + word * 64 < nnz) startBits[(size_t)blockIdx.x * kWords + word] = s;
        mine += __popcll(s);
    }
    if (lane == 0) atomicAdd(&starts, mine);
    __syncthreads();
    if (tid == 0) tileStarts[blockIdx.x] = starts;
}
static_assert(kWords <= 64 && kBlock % 64 == 0, "a lane per word of a tile");

// per virtual row: where it starts, its slice; wordBase[i] = virtual rows before the i-th word.  A workgroup takes a tile.
template <int SW>
__global__ __launch_bounds__(kBlock) void vrow_records_kernel(const unsigned long long *__restrict__ startBits, const int *__restrict__ tileBase,
                                                              const int *__restrict__ col, const int *__restrict__ ord, int nnz, int *__restrict__ wordBase,
                                                              int *__restrict__ vStart, int *__restrict__ vSlice)
{
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6, t0 = blockIdx.x * mxr::kTile, words = min(kWords, (nnz - t0 + 63) >> 6);
    const int word0 = blockIdx.x * kWords, base = tileBase[blockIdx.x];
    const unsigned long long mine = lane < words ? startBits[word0 + lane] : 0;
    int run = __popcll(mine), at = run;  // running sum over the tile's words, a lane each
#pragma unroll
    for (int off = 1; off < kWords; off <<= 1) {
        const int o = __shfl_up(run, off);
        if (lane >= off) run += o;
    }
    at = base + run - at;
    if (w == 0 && lane < words) wordBase[word0 + lane] = at;
#pragma unroll
    for (int j = 0; j < mxr::kPer; ++j) {
        const int word = j * (kBlock / 64) + w;
        const unsigned long long m = __shfl(mine, word);
        const int first = __shfl(at, word), k = t0 + word * 64 + lane;
        if (!((m >> lane) & 1)) continue;
        const int t = first + __popcll(m & ~(~0ull << lane));
        vStart[t] = k;
        vSlice[t] = col[ord ? ord[k] : k] / SW;
    }
}

// segPtr[r] = virtual rows before row r, and the row of every virtual row: a row's own thread names up to kOwnVrows of them, longer
// lists are written by the wave, one after the other.  (One row of 3 million binary64 entries, 125 thousand virtual rows: 3.4 ms by its thread alone, so 0.05.)
constexpr int kOwnVrows = 16;
__global__ __launch_bounds__(kBlock) void seg_ptr_kernel(const int *__restrict__ rowPtr, const unsigned long long *__restrict__ startBits,
                                                         const int *__restrict__ wordBase, int rows, int nnz, int nV, int *__restrict__ segPtr,
                                                         int *__restrict__ vRow)
{
    const int r = blockIdx.x * kBlock + threadIdx.x, lane = threadIdx.x & 63;
    auto before = [&](int p) { return p < nnz ? wordBase[p >> 6] + __popcll(startBits[p >> 6] & ~(~0ull << (p & 63))) : nV; };
    const int a = r < rows ? before(rowPtr[r]) : nV, e = r < rows ? before(rowPtr[r + 1]) : nV;
    if (r <= rows) segPtr[r] = a;
    const bool many = e - a > kOwnVrows;
    if (!many)
        for (int t = a; t < e; ++t) vRow[t] = r;
    for (unsigned long long m = __ballot(many); m; m &= m - 1) {
        const int l = __builtin_ctzll(m), a_ = __builtin_amdgcn_readlane(a, l), e_ = __builtin_amdgcn_readlane(e, l), r_ = __builtin_amdgcn_readlane(r, l);
        for (int t = a_ + lane; t < e_; t += 64) vRow[t] = r_;
    }
}

// the sort key of every virtual row: (slice, cap - length, kind of its row)
__global__ __launch_bounds__(kBlock) void vrow_keys_kernel(const int *__restrict__ vStart, const int *__restrict__ vRow,
                                                           const int *__restrict__ vSlice, const int *__restrict__ segPtr, int nV,
                                                           int nnz, int cap, int lightSegs, unsigned *__restrict__ key,
                                                           int *__restrict__ pay, int *__restrict__ vLen)
{
    const int t = blockIdx.x * kBlock + threadIdx.x;
    if (t >= nV) return;
    const int len = (t + 1 < nV ? vStart[t + 1] : nnz) - vStart[t];
    const int r = vRow[t], nv = segPtr[r + 1] - segPtr[r];
    const int kind = nv <= 1 ? 0 : nv <= lightSegs ? 1 : 2;
    key[t] = ((unsigned)vSlice[t] * (unsigned)(cap + 1) + (unsigned)(cap - len)) * 3u + (unsigned)kind;
    pay[t] = t;
    vLen[t] = len;
}

// segIdx[t] = 64 * chunk + lane of every virtual row
__global__ __launch_bounds__(kBlock) void vrow_places_kernel(const int *__restrict__ sorted, const int *__restrict__ chunkFirst,
                                                             const int *__restrict__ chunkN, long long chunks, int *__restrict__ segIdx)
{
    const long long i = (long long)blockIdx.x * kBlock + threadIdx.x;
    const long long c = i >> 6;
    const int l = (int)(i & 63);
    if (c >= chunks || l >= chunkN[c]) return;
    segIdx[sorted[chunkFirst[c] + l]] = (int)(c * 64 + l);
}

// every entry to its place in the streams (see DeviceSlices: lanes' column offsets of a batch
// contiguous, binary16 values likewise, binary64 values in sub-blocks of two per lane)
// (The other way round, a wave per batch that collects its 512 entries: 114 instead of 105 us for 7.6 million entries of a power law, and 520
// instead of 137 for 10.5 million binary16 entries out of order.  The entries of a chunk lie in as many rows as it has lanes, so every one
// costs its own line or two then; here they are read as they lie, and the caches put the lines of the streams together.)
template <typename V>
__global__ __launch_bounds__(kBlock) void place_entries_kernel(const unsigned long long *__restrict__ startBits, const int *__restrict__ wordBase,
                                                               const int *__restrict__ vStart, const int *__restrict__ segIdx,
                                                               const long long *__restrict__ chunkStep0, const int *__restrict__ ord,
                                                               const int *__restrict__ col, const V *__restrict__ val,
                                                               const unsigned char *__restrict__ code, int nnz, unsigned short *__restrict__ ecol,
                                                               V *__restrict__ eval, unsigned char *__restrict__ ecode)
{
    constexpr int BE = mx::kSliceBatchEntries, SW = mx::kSliceBytes / (int)sizeof(V);
    const int k = blockIdx.x * kBlock + threadIdx.x;
    if (k >= nnz) return;
    const int t = wordBase[k >> 6] + __popcll(startBits[k >> 6] & (~0ull >> (63 - (k & 63)))) - 1;  // the last that starts at or before k
    const int place = segIdx[t], l = place & 63;
    const size_t st = (size_t)chunkStep0[place >> 6] + (size_t)(k - vStart[t]), batch = st / BE, j = st % BE;
    const size_t atc = (batch * 64 + l) * BE + j;
    const size_t atv = sizeof(V) == 8 ? batch * 64 * BE + (j / 2) * 128 + (size_t)l * 2 + j % 2 : atc;
    const int p = ord ? ord[k] : k;
    ecol[atc] = (unsigned short)(col[p] & (SW - 1));
    eval[atv] = val[p];
    if (ecode) ecode[atc] = code[p];
}

// the padding of every virtual row up to its chunk's longest member names the row's own last column
template <int SW>
__global__ __launch_bounds__(kBlock) void pad_columns_kernel(const int *__restrict__ vStart, const int *__restrict__ vLen,
                                                             const int *__restrict__ segIdx,
                                                             const long long *__restrict__ chunkStep0, const int *__restrict__ chunkSteps,
                                                             const int *__restrict__ ord, const int *__restrict__ col, int nV,
                                                             unsigned short *__restrict__ ecol)
{
    constexpr int BE = mx::kSliceBatchEntries;
    const int t = blockIdx.x * kBlock + threadIdx.x;
    if (t >= nV) return;
    const int len = vLen[t], place = segIdx[t], l = place & 63, c = place >> 6;
    if (len <= 0) return;
    if (chunkSteps[c] <= len) return;
    const int k = vStart[t] + len - 1;
    const unsigned short last = (unsigned short)(col[ord ? ord[k] : k] & (SW - 1));
    for (int n = len; n < chunkSteps[c]; ++n) {
        const size_t st = (size_t)chunkStep0[c] + n, batch = st / BE, j = st % BE;
        ecol[(batch * 64 + l) * BE + j] = last;
    }
}

// rowInfo and the marks of the two lists (rows with 2..lightSegs virtual rows, rows with more).  facts[workgroup] = the most virtual
// rows of any of its rows, and of its listed rows with at most lightSegs: a word of its own, because atomics on one word take turns
// (one from every wave that had more than there was: 182 us for 700 thousand rows; so 7, and 6 in row_totals_kernel).
__global__ __launch_bounds__(kBlock) void row_info_kernel(const int *__restrict__ segPtr, const int *__restrict__ segIdx,
                                                          const char *__restrict__ elsewhere, int rows, int lightSegs,
                                                          int *__restrict__ rowInfo, int *__restrict__ isLight, int *__restrict__ isHeavy,
                                                          int2 *__restrict__ facts)
{
    __shared__ int2 part[kBlock / 64];
    const int r = blockIdx.x * kBlock + threadIdx.x;
    int n = 0, light = 0;
    if (r < rows) {
        const int a = segPtr[r];
        n = segPtr[r + 1] - a;
        const int e = elsewhere ? elsewhere[r] : 0;
        const bool fetched = e == 2;
        rowInfo[r] = fetched ? -2 : n == 0 ? (e ? -2 : -1) : n == 1 ? segIdx[a] : -2;
        const bool listed = n > 1 && !fetched;
        isLight[r] = listed && n <= lightSegs;
        isHeavy[r] = listed && n > lightSegs;
        if (listed && n <= lightSegs) light = n;
    } else if (r == rows) {  // the scans run over rows + 1 elements
        isLight[r] = isHeavy[r] = 0;
    }
    for (int off = 32; off > 0; off >>= 1) {
        n = max(n, __shfl_xor(n, off));
        light = max(light, __shfl_xor(light, off));
    }
    if ((threadIdx.x & 63) == 0) part[threadIdx.x >> 6] = int2{n, light};
    __syncthreads();
    if (threadIdx.x == 0) {
        for (int w = 1; w < kBlock / 64; ++w) {
            n = max(n, part[w].x);
            light = max(light, part[w].y);
        }
        facts[blockIdx.x] = int2{n, light};
    }
}

// What the host asks for after the row marks and their running counts, in one place: one copy instead of four.
__global__ __launch_bounds__(kBlock) void row_totals_kernel(const int2 *__restrict__ facts, int blocks, const int *__restrict__ lightPos,
                                                            const int *__restrict__ heavyPos, int rows, int *__restrict__ out)
{
    __shared__ int most, light;
    if (threadIdx.x == 0) most = light = 0;
    __syncthreads();
    int2 m = {0, 0};
#pragma unroll 4
    for (int b = threadIdx.x; b < blocks; b += kBlock) {
        m.x = max(m.x, facts[b].x);
        m.y = max(m.y, facts[b].y);
    }
    atomicMax(&most, m.x);
    atomicMax(&light, m.y);
    __syncthreads();
    if (threadIdx.x == 0) {
        out[0] = light;
        out[1] = most;
        out[2] = lightPos[rows];
        out[3] = heavyPos[rows];
    }
}

__global__ __launch_bounds__(kBlock) void row_lists_kernel(const int *__restrict__ segPtr, const int *__restrict__ segIdx,
                                                           const int *__restrict__ isLight, const int *__restrict__ isHeavy,
                                                           const int *__restrict__ lightPos, const int *__restrict__ heavyPos, int rows,
                                                           int places, int *__restrict__ lightRow, int *__restrict__ lightIdx,
                                                           int *__restrict__ heavyInfo)
{
    const int r = blockIdx.x * kBlock + threadIdx.x;
    if (r >= rows) return;
    const int a = segPtr[r], n = segPtr[r + 1] - a;
    if (isLight[r]) {
        const int i = lightPos[r];
        lightRow[i] = r;
        for (int k = 0; k < n; ++k) lightIdx[(size_t)i * places + k] = segIdx[a + k];
    }
    if (isHeavy[r]) {
        const int i = heavyPos[r];
        heavyInfo[4 * (size_t)i] = r;
        heavyInfo[4 * (size_t)i + 1] = a;
        heavyInfo[4 * (size_t)i + 2] = n;
        heavyInfo[4 * (size_t)i + 3] = 0;
    }
}

// ---- value dictionary ----
// The distinct values of a matrix (as bit patterns) and the place of the first entry that holds each, when
// there are few of them: every workgroup collects its entries' values in a table in LDS and adds what it
// found to one table in memory.  An entry costs its eight (two) bytes and a look at the LDS table -- the
// table is written only when a workgroup meets a value for the first time -- so what bounds it is reading the
// values: the plan of a constant 27-point stencil of 26.5 million binary64 entries is made in 10.7 ms, 16.7 with
// the values sorted (5.8 million binary16 entries: 6.5 and 11.9 ms).  A workgroup that meets more than `most`
// values raises the flag -- at once, also in the middle of its first entries (7.6 million distinct values: 47 us when the first thousand were gone through to the
// end and the flag was stored by all, 8 so) -- and everybody stops.  Slot kDictSlots belongs to the pattern that marks free slots.
constexpr int kDictSlots = 1024;
constexpr unsigned long long kDictFree = ~0ull;
template <typename V>
__device__ __forceinline__ unsigned long long value_bits(V v)
{
    if constexpr (sizeof(V) == 8) return __builtin_bit_cast(unsigned long long, v);
    else return __builtin_bit_cast(unsigned short, v);
}
__device__ __forceinline__ unsigned dict_hash(unsigned long long b)
{
    return (unsigned)((b * 0x9E3779B97F4A7C15ull) >> 54);  // ten bits
}
// the slot of a value in a table that holds it
__device__ __forceinline__ int dict_find(const unsigned long long *keys, unsigned long long b)
{
    if (b == kDictFree) return kDictSlots;
    unsigned h = dict_hash(b);
    for (int step = 0; step < kDictSlots && keys[h] != b; ++step) h = (h + 1) & (kDictSlots - 1);
    return (int)h;
}
// keys [kDictSlots], first [kDictSlots + 1] (INT_MAX = none), flag
template <typename V>
__global__ __launch_bounds__(kBlock) void value_set_kernel(const V *__restrict__ val, int nnz, int most, unsigned long long *__restrict__ keys,
                                                           int *__restrict__ first, int *flag)
{
    __shared__ unsigned long long keyL[kDictSlots];
    __shared__ int firstL[kDictSlots + 1];
    __shared__ int found, over, stop;  // (stop: written by one thread between two barriers, read behind the second)
    for (int i = threadIdx.x; i <= kDictSlots; i += kBlock) {
        if (i < kDictSlots) keyL[i] = kDictFree;
        firstL[i] = 0x7fffffff;
    }
    if (threadIdx.x == 0) found = over = stop = 0;
    __syncthreads();
    constexpr int E = 4;  // entries of a thread per round, all asked for before the first is looked at
    for (long long k0 = (long long)blockIdx.x * kBlock * E; k0 < nnz; k0 += (long long)gridDim.x * kBlock * E) {
        unsigned long long b[E];
#pragma unroll
        for (int j = 0; j < E; ++j) b[j] = value_bits(val[min(k0 + j * kBlock + (long long)threadIdx.x, (long long)nnz - 1)]);
#pragma unroll
        for (int j = 0; j < E; ++j) {
            const long long k = k0 + j * kBlock + threadIdx.x;
            if (k >= nnz || *(volatile int *)&found > most) continue;
            int h = kDictSlots;
            if (b[j] != kDictFree) {
                h = (int)dict_hash(b[j]);
                bool placed = false;
                for (int step = 0; step < kDictSlots && !placed; ++step) {
                    unsigned long long t = *(volatile unsigned long long *)&keyL[h];
                    if (t == kDictFree) {
                        if (*(volatile int *)&found > most) break;
                        t = atomicCAS(&keyL[h], kDictFree, b[j]);
                        if (t == kDictFree) {
                            atomicAdd(&found, 1);
                            t = b[j];
                        }
                    }
                    placed = t == b[j];
                    if (!placed) h = (h + 1) & (kDictSlots - 1);
                }
                if (!placed) {
                    over = 1;
                    continue;
                }
            }
            if ((int)k < *(volatile int *)&firstL[h]) atomicMin(&firstL[h], (int)k);
        }
        __syncthreads();
        if (threadIdx.x == 0 && (over || found > most || *(volatile int *)flag)) {
            stop = 1;
            if (*(volatile int *)flag == 0) *(volatile int *)flag = 1;  // (stores to one word take turns)
        }
        __syncthreads();
        if (stop) return;
    }
    for (int i = threadIdx.x; i <= kDictSlots; i += kBlock) {
        const int f = firstL[i];
        if (f == 0x7fffffff) continue;
        unsigned h = kDictSlots;
        if (i < kDictSlots) {
            h = dict_hash(keyL[i]);
            bool placed = false;
            for (int step = 0; step < kDictSlots && !placed; ++step) {
                const unsigned long long t = atomicCAS(&keys[h], kDictFree, keyL[i]);
                placed = t == kDictFree || t == keyL[i];
                if (!placed) h = (h + 1) & (kDictSlots - 1);
            }
            if (!placed) {  // more than kDictSlots values among all workgroups
                *(volatile int *)flag = 1;
                continue;
            }
        }
        atomicMin(&first[h], f);
    }
}
__global__ __launch_bounds__(kBlock) void dict_clear_kernel(unsigned long long *__restrict__ keys, int *__restrict__ first, int *__restrict__ flag)
{
    for (int i = threadIdx.x; i <= kDictSlots; i += kBlock) {
        if (i < kDictSlots) keys[i] = kDictFree;
        first[i] = 0x7fffffff;
    }
    if (threadIdx.x == 0) *flag = 0;
}
// code of every entry: what `codeOf` says of the slot of its value
template <typename V>
__global__ __launch_bounds__(kBlock) void value_codes_kernel(const V *__restrict__ val, int nnz, const unsigned long long *__restrict__ keys,
                                                             const unsigned char *__restrict__ codeOf, unsigned char *__restrict__ code)
{
    __shared__ unsigned long long keyL[kDictSlots];
    __shared__ unsigned char codeL[kDictSlots + 1];
    for (int i = threadIdx.x; i <= kDictSlots; i += kBlock) {
        if (i < kDictSlots) keyL[i] = keys[i];
        codeL[i] = codeOf[i];
    }
    __syncthreads();
    // (four consecutive entries per thread and round, their codes in one store)
    for (long long k = ((long long)blockIdx.x * kBlock + threadIdx.x) * 4; k < nnz; k += (long long)gridDim.x * kBlock * 4) {
        unsigned w = 0;
#pragma unroll
        for (int j = 0; j < 4; ++j)
            if (k + j < nnz) w |= (unsigned)codeL[dict_find(keyL, value_bits(val[k + j]))] << (8 * j);
        if (k + 4 <= nnz) *(unsigned *)(code + k) = w;
        else
            for (int j = 0; j < 4 && k + j < nnz; ++j) code[k + j] = (unsigned char)(w >> (8 * j));
    }
}

// ---- statistics and the row-tile form from device arrays ----
// bad |= 1 unless rowPtr rises from 0 to nnz; bad |= 2 for a column outside [0, cols)
__global__ __launch_bounds__(kBlock) void check_csr_kernel(const int *__restrict__ rowPtr, const int *__restrict__ col, int rows, int cols,
                                                           int nnz, int *__restrict__ bad)
{
    const long long i = (long long)blockIdx.x * kBlock + threadIdx.x;
    if (i <= rows) {
        const int p = rowPtr[i];
        if ((i == 0 && p != 0) || (i == rows && p != nnz) || (i < rows && rowPtr[i + 1] < p) || p < 0 || p > nnz) atomicOr(bad, 1);
    }
    if (i < nnz && (unsigned)col[i] >= (unsigned)cols) atomicOr(bad, 2);
}
// sum += distinct 64-byte lines of x that the 64 entries of every stride-th window name: a lane per entry, which counts
// when no lane below it has its line.  The lanes with a lane's line are found bit by bit, one ballot for each that differs in the wave (compared
// with the other lanes' lines in turn instead: 84 us for the 118 thousand windows of 7.6 million entries; so 40).  One atomic per workgroup.
constexpr int kLinesBlocks = 2048;
__global__ __launch_bounds__(kBlock) void window_lines_kernel(const int *__restrict__ col, long long sampled, long long stride, int perLine,
                                                              unsigned long long *__restrict__ sum)
{
    __shared__ int part[kBlock / 64];
    const int lane = threadIdx.x & 63, waves = gridDim.x * (kBlock / 64);
    int d = 0;
    long long i = (blockIdx.x * kBlock + threadIdx.x) >> 6;
    int c = i < sampled ? col[i * stride * 64 + lane] : 0;
    for (; i < sampled; i += waves) {
        const int line = c / perLine;
        c = col[min(i + waves, sampled - 1) * stride * 64 + lane];  // (the next window's, on its way meanwhile)
        const unsigned x = (unsigned)(line ^ __builtin_amdgcn_readfirstlane(line));
        unsigned lo = ~0u, hi = ~0u, done = 0;
        // (a bit that differs among the lanes, then the next)
        for (unsigned long long any = __ballot(x != 0); any; any = __ballot((x & ~done) != 0)) {
            const unsigned one = (unsigned)__builtin_amdgcn_readlane((int)(x & ~done), __builtin_ctzll(any)), bit = one & (0u - one);
            const unsigned set = (x & bit) ? ~0u : 0u;
            const unsigned long long b = __ballot(set != 0);
            lo &= ~((unsigned)b ^ set);
            hi &= ~((unsigned)(b >> 32) ^ set);
            done |= bit;
        }
        const int below = __builtin_amdgcn_mbcnt_hi(hi, __builtin_amdgcn_mbcnt_lo(lo, 0));
        d += __popcll(__ballot(below == 0));
    }
    if (lane == 0) part[threadIdx.x >> 6] = d;
    __syncthreads();
    if (threadIdx.x == 0) {
        unsigned long long v = 0;
        for (int w = 0; w < kBlock / 64; ++w) v += (unsigned)part[w];
        atomicAdd(sum, v);
    }
}
// one wave per workgroup of the row kernel: the lowest and the highest column of its entries
__global__ __launch_bounds__(kBlock) void block_ranges_kernel(const int4 *__restrict__ desc, const int *__restrict__ col, int nBlocks,
                                                              int *__restrict__ lo, int *__restrict__ wide)
{
    const int b = (blockIdx.x * kBlock + threadIdx.x) >> 6, lane = threadIdx.x & 63;
    if (b >= nBlocks) return;
    const int4 d = desc[b];
    int mn = 0x7fffffff, mx_ = 0;
    for (int p = d.z + lane; p < d.w; p += 64) {
        mn = min(mn, col[p]);
        mx_ = max(mx_, col[p]);
    }
    for (int o = 32; o > 0; o >>= 1) {
        mn = min(mn, __shfl_xor(mn, o, 64));
        mx_ = max(mx_, __shfl_xor(mx_, o, 64));
    }
    if (lane == 0) {
        lo[b] = d.w > d.z ? mn : 0;
        if (d.w > d.z && mx_ - mn > 65535) atomicOr(wide, 1);
    }
}
__global__ __launch_bounds__(kBlock) void narrow_columns_kernel(const int4 *__restrict__ desc, const int *__restrict__ col,
                                                                const int *__restrict__ lo, int nBlocks, unsigned short *__restrict__ c16)
{
    const int b = (blockIdx.x * kBlock + threadIdx.x) >> 6, lane = threadIdx.x & 63;
    if (b >= nBlocks) return;
    const int4 d = desc[b];
    const int base = lo[b];
    for (int p = d.z + lane; p < d.w; p += 64) c16[p] = (unsigned short)(col[p] - base);
}

}  // namespace mxl

namespace mx {

// The value dictionary of a matrix in device memory, as make_value_dict gives it on the host: at
// most 255 distinct bit patterns, numbered in the order of their first entry; codes[nnz] (device)
// and dict (256 values, host, zero-padded).  *nDict = 0 when the matrix has more.
template <typename V>
static int device_value_dict(const V *val, int nnz, mxl::Buf &codes, std::vector<unsigned char> &dict, int *nDict, hipStream_t s,
                             int most = 255, size_t codePad = 0)
{
    using namespace mxl;
    *nDict = 0;
    Buf table;  // keys, codes of the slots, first places, flag
    const size_t keyB = kDictSlots * 8, codeB = 2048, firstB = (kDictSlots + 1) * 4;
    MXL_TRY(mx::dev_malloc(&table.p, keyB + codeB + firstB + 256));
    unsigned long long *keys = table.as<unsigned long long>();
    unsigned char *codeOf = table.as<unsigned char>() + keyB;
    int *first = (int *)(codeOf + codeB), *flag = first + kDictSlots + 1;
    struct Host {
        unsigned long long keys[kDictSlots];
        unsigned char codeOf[2048];
        int first[kDictSlots + 1], flag;
    };
    static_assert(sizeof(Host) == kDictSlots * 8 + 2048 + (kDictSlots + 2) * 4, "the table comes down in one copy");
    std::vector<Host> hv(1);
    Host &h = hv[0];
    hipLaunchKernelGGL(dict_clear_kernel, dim3(1), dim3(kBlock), 0, s, keys, first, flag);
    hipLaunchKernelGGL(value_set_kernel<V>, dim3((unsigned)std::min<long long>(1024, ((long long)nnz + 1023) / 1024)), dim3(kBlock), 0, s, val, nnz,
                       most, keys, first, flag);
    MXL_TRY(hipGetLastError());
    MXL_TRY(hipMemcpyAsync(&h, table.p, sizeof(Host), hipMemcpyDeviceToHost, s));
    MXL_TRY(hipStreamSynchronize(s));
    if (h.flag) return MX_OK;
    std::vector<int> order;
    for (int i = 0; i <= kDictSlots; ++i)
        if (h.first[i] != 0x7fffffff) order.push_back(i);
    const int nd = (int)order.size();
    if (nd > most) return MX_OK;
    // codes in the order of first appearance, as the host's scan over the entries numbers them
    std::sort(order.begin(), order.end(), [&](int a, int b) { return h.first[a] < h.first[b]; });
    std::memset(h.codeOf, 0, sizeof(h.codeOf));
    dict.assign((size_t)256 * sizeof(V), 0);
    for (int c = 0; c < nd; ++c) {
        h.codeOf[order[c]] = (unsigned char)c;
        const unsigned long long v = order[c] < kDictSlots ? h.keys[order[c]] : kDictFree;
        std::memcpy(&dict[(size_t)c * sizeof(V)], &v, sizeof(V));  // little-endian: the low bytes are the value
    }
    MXL_TRY(hipMemcpyAsync(codeOf, h.codeOf, sizeof(h.codeOf), hipMemcpyHostToDevice, s));
    MXL_TRY(mx::dev_malloc(&codes.p, (size_t)nnz + codePad));
    if (codePad) MXL_TRY(hipMemsetAsync((unsigned char *)codes.p + nnz, 0, codePad, s));
    hipLaunchKernelGGL(value_codes_kernel<V>, dim3((unsigned)std::min<long long>(4096, ((long long)nnz + 1023) / 1024)), dim3(kBlock), 0, s, val, nnz,
                       (const unsigned long long *)keys, (const unsigned char *)codeOf, codes.as<unsigned char>());
    MXL_TRY(hipGetLastError());
    MXL_TRY(hipStreamSynchronize(s));
    *nDict = nd;
    return MX_OK;
}

int value_dict_device(mx_dtype dtype, const void *val_dev, int nnz, int most, void **codes, std::vector<unsigned char> &dict, int *nDict,
                      hipStream_t s)
{
    mxl::Buf c;
    *codes = nullptr;
    const int rc = dtype == MX_F64 ? device_value_dict<double>((const double *)val_dev, nnz, c, dict, nDict, s, most)
                                   : device_value_dict<_Float16>((const _Float16 *)val_dev, nnz, c, dict, nDict, s, most);
    if (rc == MX_OK) *codes = c.take();
    return rc;
}

template <typename V>
static int build_slices_device_t(mx_dtype dtype, int rows, int cols, int nnz, const int *rowPtr, const int *col, const V *val, int nCU,
                                 int S, const char *elsewhere, DeviceSlices &D, hipStream_t s, std::vector<int> *segPtrOut,
                                 std::vector<int> *segIdxOut, int fused)
{
    using namespace mxl;
    const int E = slice_step_entries(dtype), BE = kSliceBatchEntries, SW = slice_cols(dtype), W = kSliceWaves;
    const int budget = std::max(nCU, 1);
    const long long fair = (long long)nnz / ((long long)budget * W * 64);
    int cap = (int)std::min<long long>(512, std::max<long long>(16, (fair + BE - 1) / BE * BE));
    if (const int v = mx::opt().slice_cap)
        if (v >= BE && v <= 4096) cap = v / BE * BE;
    D = DeviceSlices();
    D.S = S;
    D.rows = rows;
    D.cols = cols;
    D.sliceCols = SW;
    D.nnz = nnz;
    // ---- virtual rows, from the entries as they lie; where some row's columns are not ascending, from their order
    Buf ordBuf, flag, startBits, tileStarts, tileBase, wordBase;
    const size_t tiles = ((size_t)nnz + mxr::kTile - 1) / mxr::kTile, words = ((size_t)nnz + 63) / 64;
    MXL_TRY(mx::dev_malloc(&flag.p, 256));
    MXL_TRY(mx::dev_malloc(&startBits.p, (words + 1) * 8));
    MXL_TRY(mx::dev_malloc(&tileStarts.p, (tiles + 1) * 4));
    MXL_TRY(mx::dev_malloc(&tileBase.p, (tiles + 1) * 4));
    MXL_TRY(mx::dev_malloc(&wordBase.p, (words + 1) * 4));
    MXL_TRY(hipMemsetAsync(flag.p, 0, 256, s));
    MXL_TRY(hipMemsetAsync(tileStarts.as<int>() + tiles, 0, 4, s));
    Buf tmp;
    size_t scanBytes = 0;
    const size_t nScan = std::max(tiles, (size_t)rows + 1) + 1;
    MXL_TRY(rocprim::exclusive_scan(nullptr, scanBytes, (const int *)nullptr, (int *)nullptr, 0, nScan, rocprim::plus<int>(), s));
    MXL_TRY(mx::dev_malloc(&tmp.p, scanBytes + 256));
    constexpr int SliceCols = kSliceBytes / (int)sizeof(V);
    const int *ord = nullptr;
    int nV = 0;
    auto find_vrows = [&](int *unsorted) -> int {
        int got = 0;
        hipLaunchKernelGGL(vrow_starts_kernel<SliceCols>, mxr::tile_grid(nnz), dim3(kBlock), 0, s, rowPtr, col, ord, rows, nnz, cap,
                           startBits.as<unsigned long long>(), tileStarts.as<int>(), flag.as<int>());
        MXL_TRY(hipGetLastError());
        MXL_TRY(rocprim::exclusive_scan(tmp.p, scanBytes, (const int *)tileStarts.p, tileBase.as<int>(), 0, tiles + 1, rocprim::plus<int>(), s));
        MXL_TRY(hipMemcpyAsync(&nV, tileBase.as<int>() + tiles, 4, hipMemcpyDeviceToHost, s));
        MXL_TRY(hipMemcpyAsync(&got, flag.p, 4, hipMemcpyDeviceToHost, s));
        MXL_TRY(hipStreamSynchronize(s));
        *unsorted = got;
        return MX_OK;
    };
    int unsorted = 0, rc;
    if (nnz > 0 && (rc = find_vrows(&unsorted))) return rc;
    if (unsorted) {
        // inside a workgroup per row or group of rows, where there is no row too long for that
        // (15.8 million entries in a million rows: keys and radix sort 0.91 ms, so 0.39)
        Buf list;
        mxs::RowClasses classes{};
        int *count = flag.as<int>() + 8;
        MXL_TRY(mx::dev_malloc(&ordBuf.p, (size_t)nnz * 4));
        MXL_TRY(mx::dev_malloc(&list.p, mxs::list_ints(nnz) * 4));
        MXL_TRY(mxs::classify_rows(rowPtr, rows, nnz, list.as<int>(), count, s));
        MXL_TRY(hipMemcpyAsync(classes.n, count, sizeof(classes.n), hipMemcpyDeviceToHost, s));
        MXL_TRY(hipStreamSynchronize(s));
        if (classes.n[mxs::kClasses] == 0) {
            MXL_TRY(mxs::sort_rows(rowPtr, rows, nnz, list.as<int>(), classes, RowColumns{col, ordBuf.as<int>()}, s));
        } else {
            int colBits = 1, rowBits = 1;
            while (colBits < 31 && (1ll << colBits) < (long long)cols) ++colBits;
            while (rowBits < 31 && (1ll << rowBits) < (long long)rows) ++rowBits;
            Buf keyIn, keyOut, payIn, tmp;
            size_t sortBytes = 0;
            MXL_TRY(rocprim::radix_sort_pairs(nullptr, sortBytes, (const unsigned long long *)nullptr, (unsigned long long *)nullptr,
                                              (const int *)nullptr, (int *)nullptr, (size_t)nnz, 0u, (unsigned)(colBits + rowBits), s));
            MXL_TRY(mx::dev_malloc(&keyIn.p, (size_t)nnz * 8));
            MXL_TRY(mx::dev_malloc(&keyOut.p, (size_t)nnz * 8));
            MXL_TRY(mx::dev_malloc(&payIn.p, (size_t)nnz * 4));
            MXL_TRY(mx::dev_malloc(&tmp.p, sortBytes + 256));
            hipLaunchKernelGGL(sort_keys_kernel, mxr::tile_grid(nnz), dim3(kBlock), 0, s, rowPtr, col, rows, nnz, colBits,
                               keyIn.as<unsigned long long>(), payIn.as<int>());
            MXL_TRY(hipGetLastError());
            MXL_TRY(rocprim::radix_sort_pairs(tmp.p, sortBytes, (const unsigned long long *)keyIn.p, keyOut.as<unsigned long long>(),
                                              (const int *)payIn.p, ordBuf.as<int>(), (size_t)nnz, 0u, (unsigned)(colBits + rowBits), s));
        }
        ord = ordBuf.as<int>();
        if ((rc = find_vrows(&unsorted))) return rc;
    }
    D.vrows = nV;
    Buf vStart, vRow, vSlice, vLen, segPtr, key, keyOut, pay, sorted;
    const size_t nv1 = (size_t)nV + 1;
    MXL_TRY(mx::dev_malloc(&vStart.p, nv1 * 4));
    MXL_TRY(mx::dev_malloc(&vRow.p, nv1 * 4));
    MXL_TRY(mx::dev_malloc(&vSlice.p, nv1 * 4));
    MXL_TRY(mx::dev_malloc(&vLen.p, nv1 * 4));
    MXL_TRY(mx::dev_malloc(&segPtr.p, ((size_t)rows + 2) * 4));
    MXL_TRY(mx::dev_malloc(&key.p, nv1 * 4));
    MXL_TRY(mx::dev_malloc(&keyOut.p, nv1 * 4));
    MXL_TRY(mx::dev_malloc(&pay.p, nv1 * 4));
    MXL_TRY(mx::dev_malloc(&sorted.p, nv1 * 4));
    const unsigned long long *bits = startBits.as<unsigned long long>();
    if (nnz > 0) {
        hipLaunchKernelGGL(vrow_records_kernel<SliceCols>, mxr::tile_grid(nnz), dim3(kBlock), 0, s, bits, (const int *)tileBase.p, col, ord, nnz,
                           wordBase.as<int>(), vStart.as<int>(), vSlice.as<int>());
        MXL_TRY(hipGetLastError());
    }
    hipLaunchKernelGGL(seg_ptr_kernel, grid((long long)rows + 1), dim3(kBlock), 0, s, rowPtr, bits, (const int *)wordBase.p, rows, nnz, nV,
                       segPtr.as<int>(), vRow.as<int>());
    MXL_TRY(hipGetLastError());
    if (nV > 0) {
        hipLaunchKernelGGL(vrow_keys_kernel, grid(nV), dim3(kBlock), 0, s, (const int *)vStart.p, (const int *)vRow.p, (const int *)vSlice.p,
                           (const int *)segPtr.p, nV, nnz, cap, kSliceLightSegs, key.as<unsigned>(), pay.as<int>(), vLen.as<int>());
        MXL_TRY(hipGetLastError());
    }
    // ---- the one-launch form, where it is wanted and the matrix suits it (on the host where there are few virtual rows, or its digits
    // are too many for the device: their records come down, the plan goes up)
    ChunkPlan C;
    FusedPlan F;
    if (fused && nV > 0 && !elsewhere && fused_plan_on_device(S, cap, nV)) {
        bool taken = false;
        const int rc = plan_fused_device(dtype, budget, S, rows, nnz, cap, nV, fused, rowPtr, (const int *)segPtr.p, (const int *)vRow.p, (const int *)vSlice.p,
                                         (const int *)vLen.p, sorted.as<int>(), C, F, &taken, s);
        if (rc) return rc;
        if (!taken) {
            C.made.release();
            F.wgGroups.release();
        }
        D.fused = taken;
        fused = 0;
    }
    SlicePlan SP;
    int fusedPlaces = 0;
    bool fusedTaken = false;  // (by the host's plan; D.fused: by the device's)
    std::vector<int> hSegPtr;
    if (fused && nV > 0 && !elsewhere) {
        std::vector<int> hRowPtr((size_t)rows + 1), hSlice((size_t)nV), hLen((size_t)nV), hSorted;
        hSegPtr.resize((size_t)rows + 1);
        MXL_TRY(hipMemcpyAsync(hRowPtr.data(), rowPtr, ((size_t)rows + 1) * 4, hipMemcpyDeviceToHost, s));
        MXL_TRY(hipMemcpyAsync(hSegPtr.data(), segPtr.p, ((size_t)rows + 1) * 4, hipMemcpyDeviceToHost, s));
        MXL_TRY(hipMemcpyAsync(hSlice.data(), vSlice.p, (size_t)nV * 4, hipMemcpyDeviceToHost, s));
        MXL_TRY(hipMemcpyAsync(hLen.data(), vLen.p, (size_t)nV * 4, hipMemcpyDeviceToHost, s));
        MXL_TRY(hipStreamSynchronize(s));
        const int rc = plan_fused_records(dtype, budget, S, rows, cap, hRowPtr.data(), hSegPtr.data(), hSlice.data(), hLen.data(), nV, fused,
                                          hSorted, SP, &fusedPlaces);
        if (rc < 0) return rc;
        fusedTaken = rc == 1;
        if (fusedTaken) {
            MXL_TRY(hipMemcpyAsync(sorted.p, hSorted.data(), (size_t)nV * 4, hipMemcpyHostToDevice, s));
            MXL_TRY(hipStreamSynchronize(s));  // `hSorted` leaves scope
        }
    }
    if (nV > 0 && !fusedTaken && !D.fused) {
        unsigned keyBits = 1;
        while (keyBits < 32 && (1ull << keyBits) < (unsigned long long)S * (unsigned long long)(cap + 1) * 3ull) ++keyBits;
        size_t sortBytes = 0;
        MXL_TRY(rocprim::radix_sort_pairs(nullptr, sortBytes, (const unsigned *)nullptr, (unsigned *)nullptr, (const int *)nullptr,
                                          (int *)nullptr, (size_t)nV, 0u, keyBits, s));
        Buf sortTmp;
        MXL_TRY(mx::dev_malloc(&sortTmp.p, sortBytes + 256));
        MXL_TRY(rocprim::radix_sort_pairs(sortTmp.p, sortBytes, (const unsigned *)key.p, keyOut.as<unsigned>(), (const int *)pay.p,
                                          sorted.as<int>(), (size_t)nV, 0u, keyBits, s));
    }
    // ---- chunks: which workgroup and wave streams which
    auto up = [&](void **dst, const void *src, size_t bytes) -> int {
        MXL_TRY(mx::dev_malloc(dst, std::max<size_t>(bytes, 4)));
        if (bytes) MXL_TRY(hipMemcpyAsync(*dst, src, bytes, hipMemcpyHostToDevice, s));
        return MX_OK;
    };
    Buf chunkFirst, chunkN, chunkSteps, chunkStep0;
    if (fusedTaken) {
        C.nWG = SP.nWG;
        C.maxWgChunks = SP.maxWgChunks;
        C.totalSteps = SP.totalSteps;
        C.totalChunks = SP.totalChunks;
        if ((rc = up(&C.wgDesc.p, SP.wgDesc.data(), SP.wgDesc.size() * 4))) return rc;
        if ((rc = up(&C.waveDesc.p, SP.waveDesc.data(), SP.waveDesc.size() * 4))) return rc;
        if ((rc = up(&C.chunkEnd.p, SP.chunkEnd.data(), SP.chunkEnd.size() * 4))) return rc;
        if ((rc = up(&chunkFirst.p, SP.chunkFirst.data(), SP.chunkFirst.size() * 4))) return rc;
        if ((rc = up(&chunkN.p, SP.chunkN.data(), SP.chunkN.size() * 4))) return rc;
        if ((rc = up(&chunkSteps.p, SP.chunkSteps.data(), SP.chunkSteps.size() * 4))) return rc;
        if ((rc = up(&chunkStep0.p, SP.chunkStep0.data(), SP.chunkStep0.size() * 8))) return rc;
        C.chunkFirst = chunkFirst.as<int>();
        C.chunkN = chunkN.as<int>();
        C.chunkSteps = chunkSteps.as<int>();
        C.chunkStep0 = chunkStep0.as<long long>();
    } else if (!D.fused) {
        if ((rc = plan_chunks_device(dtype, budget, S, nV, (const unsigned *)keyOut.p, (unsigned)(cap + 1) * 3u, (const int *)sorted.p, (const int *)vLen.p, C, s)))
            return rc;
    }
    D.wgDesc = (int *)C.wgDesc.take();
    D.waveDesc = (int *)C.waveDesc.take();
    D.chunkEnd = (int *)C.chunkEnd.take();
    D.nWG = C.nWG;
    D.maxWgChunks = C.maxWgChunks;
    D.steps = C.totalSteps;
    D.chunks = C.totalChunks;
    // ---- the streams
    const size_t nEcol = ((size_t)C.totalSteps + kSlicePadSteps) * 64 * E;
    MXL_TRY(mx::dev_malloc((void **)&D.ecol, nEcol * 2));
    MXL_TRY(hipMemsetAsync(D.ecol, 0, nEcol * 2, s));
    MXL_TRY(mx::dev_malloc(&D.eval, nEcol * sizeof(V)));
    MXL_TRY(hipMemsetAsync(D.eval, 0, nEcol * sizeof(V), s));
    Buf codes;
    std::vector<unsigned char> dict;
    int nDict = 0;
    {
        if (nnz >= 65536 && mx::opt().csr_dict != 0) {
            if ((rc = device_value_dict<V>(val, nnz, codes, dict, &nDict, s))) return rc;
        }
        if (nDict > 0) {
            MXL_TRY(mx::dev_malloc((void **)&D.ecode, nEcol));
            MXL_TRY(hipMemsetAsync(D.ecode, 255, nEcol, s));
            if ((rc = up(&D.dict, dict.data(), dict.size()))) return rc;
            D.nDict = nDict;
        }
    }
    MXL_TRY(mx::dev_malloc((void **)&D.segIdx, nv1 * 4));
    MXL_TRY(hipMemsetAsync(D.segIdx, 0, nv1 * 4, s));
    if (C.totalChunks > 0) {
        hipLaunchKernelGGL(vrow_places_kernel, grid(C.totalChunks * 64), dim3(kBlock), 0, s, (const int *)sorted.p, C.chunkFirst,
                           C.chunkN, C.totalChunks, D.segIdx);
        MXL_TRY(hipGetLastError());
    }
    if (nnz > 0) {
        hipLaunchKernelGGL(place_entries_kernel<V>, grid(nnz), dim3(kBlock), 0, s, bits, (const int *)wordBase.p, (const int *)vStart.p,
                           (const int *)D.segIdx, C.chunkStep0, ord, col, val, (const unsigned char *)codes.p, nnz, D.ecol, (V *)D.eval,
                           nDict > 0 ? D.ecode : nullptr);
        MXL_TRY(hipGetLastError());
        hipLaunchKernelGGL(pad_columns_kernel<SliceCols>, grid(nV), dim3(kBlock), 0, s, (const int *)vStart.p, (const int *)vLen.p, (const int *)D.segIdx,
                           C.chunkStep0, C.chunkSteps, ord, col, nV, D.ecol);
        MXL_TRY(hipGetLastError());
    }
    // ---- how the sums become y
    const size_t nInfo = ((size_t)rows + 3) / 4 * 4 + 4;
    MXL_TRY(mx::dev_malloc((void **)&D.rowInfo, nInfo * 4));
    MXL_TRY(hipMemsetAsync(D.rowInfo, 0xfe, nInfo * 4, s));  // (overwritten below for the rows; the padding must read -2)
    {
        std::vector<int> fill(nInfo - (size_t)rows, -2);
        MXL_TRY(hipMemcpyAsync(D.rowInfo + rows, fill.data(), fill.size() * 4, hipMemcpyHostToDevice, s));
        MXL_TRY(hipStreamSynchronize(s));  // `fill` leaves scope
    }
    Buf isLight, isHeavy, lightPos, heavyPos, facts;
    const size_t r1 = (size_t)rows + 1;
    const int rowBlocks = (int)(((long long)rows + kBlock) / kBlock);
    MXL_TRY(mx::dev_malloc(&facts.p, (size_t)rowBlocks * 8));
    MXL_TRY(mx::dev_malloc(&isLight.p, r1 * 4));
    MXL_TRY(mx::dev_malloc(&isHeavy.p, r1 * 4));
    MXL_TRY(mx::dev_malloc(&lightPos.p, r1 * 4));
    MXL_TRY(mx::dev_malloc(&heavyPos.p, r1 * 4));
    hipLaunchKernelGGL(row_info_kernel, dim3((unsigned)rowBlocks), dim3(kBlock), 0, s, (const int *)segPtr.p, (const int *)D.segIdx, elsewhere,
                       rows, kSliceLightSegs, D.rowInfo, isLight.as<int>(), isHeavy.as<int>(), facts.as<int2>());
    MXL_TRY(hipGetLastError());
    MXL_TRY(rocprim::exclusive_scan(tmp.p, scanBytes, (const int *)isLight.p, lightPos.as<int>(), 0, r1, rocprim::plus<int>(), s));
    MXL_TRY(rocprim::exclusive_scan(tmp.p, scanBytes, (const int *)isHeavy.p, heavyPos.as<int>(), 0, r1, rocprim::plus<int>(), s));
    int got[4] = {0, 0, 0, 0};
    hipLaunchKernelGGL(row_totals_kernel, dim3(1), dim3(kBlock), 0, s, (const int2 *)facts.p, rowBlocks, (const int *)lightPos.p, (const int *)heavyPos.p, rows,
                       flag.as<int>() + 16);
    MXL_TRY(hipGetLastError());
    MXL_TRY(hipMemcpyAsync(got, flag.as<int>() + 16, sizeof(got), hipMemcpyDeviceToHost, s));
    MXL_TRY(hipStreamSynchronize(s));
    const int mostLight = got[0], mostVrows = got[1], nLight = got[2], nHeavy = got[3];
    D.nLight = nLight;
    D.nHeavy = nHeavy;
    D.mostVrows = std::max(mostVrows, nV > 0 ? 1 : 0);
    const int places = mostLight > 4 ? kSliceLightSegs : 4;
    D.lightQuads = places / 4;
    MXL_TRY(mx::dev_malloc((void **)&D.lightRow, ((size_t)nLight + 1) * 4));
    MXL_TRY(hipMemsetAsync(D.lightRow, 0, ((size_t)nLight + 1) * 4, s));
    MXL_TRY(mx::dev_malloc((void **)&D.lightIdx, ((size_t)nLight * places + 8) * 4));
    MXL_TRY(hipMemsetAsync(D.lightIdx, 0xff, (size_t)nLight * places * 4, s));                    // -1 = no virtual row
    MXL_TRY(hipMemsetAsync(D.lightIdx + (size_t)nLight * places, 0, 8 * 4, s));                   // the spare entries read 0
    MXL_TRY(mx::dev_malloc((void **)&D.heavyInfo, ((size_t)nHeavy * 4 + 4) * 4));
    MXL_TRY(hipMemsetAsync(D.heavyInfo, 0, ((size_t)nHeavy * 4 + 4) * 4, s));
    hipLaunchKernelGGL(row_lists_kernel, grid(rows), dim3(kBlock), 0, s, (const int *)segPtr.p, (const int *)D.segIdx, (const int *)isLight.p,
                       (const int *)isHeavy.p, (const int *)lightPos.p, (const int *)heavyPos.p, rows, places, D.lightRow, D.lightIdx,
                       D.heavyInfo);
    MXL_TRY(hipGetLastError());
    const size_t accBytes = dtype == MX_F64 ? 8 : 4;
    MXL_TRY(mx::dev_malloc(&D.partial, ((size_t)C.totalChunks * 64 + 64) * accBytes));
    MXL_TRY(hipMemsetAsync(D.partial, 0, ((size_t)C.totalChunks * 64 + 64) * accBytes, s));
    if (fusedTaken || D.fused) {
        // what the one-launch kernel needs beyond the two-launch arrays (which stay valid: the plan falls back on them)
        const size_t nTarget = (size_t)C.totalChunks * 64 + 64;  // (64 spare entries, zero)
        if (D.fused) {
            D.nGroups = F.nGroups;
            D.maxWgGroups = F.maxWgGroups;
            D.placesPerRow = F.places;
            D.wgGroups = (int *)F.wgGroups.take();
            D.groupNeed = (int *)F.groupNeed.take();
            MXL_TRY(mx::dev_malloc((void **)&D.fusedTarget, nTarget * 4));
            if ((rc = fused_targets_device(F.nGroups, F.places, C.totalChunks, (const int *)segPtr.p, D.segIdx, (const int *)vRow.p, nV, D.fusedTarget, s)))
                return rc;
        } else {
            std::vector<int> hSegIdx(nv1, 0), target;
            MXL_TRY(hipMemcpyAsync(hSegIdx.data(), D.segIdx, nv1 * 4, hipMemcpyDeviceToHost, s));
            MXL_TRY(hipStreamSynchronize(s));
            fused_targets(rows, SP.nGroups, fusedPlaces, SP.totalChunks, hSegPtr.data(), hSegIdx.data(), target);
            D.nGroups = SP.nGroups;
            D.maxWgGroups = SP.maxWgGroups;
            D.placesPerRow = fusedPlaces;
            if ((rc = up((void **)&D.wgGroups, SP.wgGroups.data(), SP.wgGroups.size() * 4))) return rc;
            if ((rc = up((void **)&D.groupNeed, SP.groupNeed.data(), SP.groupNeed.size() * 4))) return rc;
            MXL_TRY(mx::dev_malloc((void **)&D.fusedTarget, nTarget * 4));
            MXL_TRY(hipMemsetAsync(D.fusedTarget, 0, nTarget * 4, s));
            MXL_TRY(hipMemcpyAsync(D.fusedTarget, target.data(), target.size() * 4, hipMemcpyHostToDevice, s));
            MXL_TRY(hipStreamSynchronize(s));  // `target` leaves scope
        }
        const size_t nCount = (size_t)D.nGroups + 1, nClaim = (size_t)C.nWG + 1;
        const size_t sumBytes = ((size_t)D.nGroups * D.placesPerRow * kFusedGroupRows + 64) * accBytes;
        MXL_TRY(mx::dev_malloc((void **)&D.groupCount, nCount * 4));
        MXL_TRY(hipMemsetAsync(D.groupCount, 0, nCount * 4, s));
        MXL_TRY(mx::dev_malloc((void **)&D.claim, nClaim * 4));
        MXL_TRY(hipMemsetAsync(D.claim, 0, nClaim * 4, s));
        MXL_TRY(mx::dev_malloc(&D.fusedSums, sumBytes));
        MXL_TRY(hipMemsetAsync(D.fusedSums, 0, sumBytes, s));
        D.fused = true;
    }
    if (segPtrOut) {
        segPtrOut->assign((size_t)rows + 1, 0);
        MXL_TRY(hipMemcpyAsync(segPtrOut->data(), segPtr.p, ((size_t)rows + 1) * 4, hipMemcpyDeviceToHost, s));
    }
    if (segIdxOut) {
        segIdxOut->assign(nv1, 0);
        MXL_TRY(hipMemcpyAsync(segIdxOut->data(), D.segIdx, nv1 * 4, hipMemcpyDeviceToHost, s));
    }
    MXL_TRY(hipStreamSynchronize(s));
    return MX_OK;
}

int check_csr_device(int rows, int cols, int nnz, const int *rowPtr_dev, const int *col_dev, hipStream_t s, const char *who)
{
    using namespace mxl;
    // (the kernels number entries and rows with 32-bit thread indices, rounded up to whole workgroups)
    constexpr int most = 2147483647 - 2 * kBlock;
    if (rows > most || cols > most || nnz > most) {
        set_error(std::string(who) + ": more rows, columns or entries than the device route can number");
        return MX_ERR_ARG;
    }
    Buf bad;
    MXL_TRY(mx::dev_malloc(&bad.p, 256));
    MXL_TRY(hipMemsetAsync(bad.p, 0, 256, s));
    hipLaunchKernelGGL(check_csr_kernel, grid(std::max<long long>((long long)rows + 1, nnz)), dim3(kBlock), 0, s, rowPtr_dev, col_dev, rows,
                       cols, nnz, bad.as<int>());
    MXL_TRY(hipGetLastError());
    int h = 0;
    MXL_TRY(hipMemcpyAsync(&h, bad.p, 4, hipMemcpyDeviceToHost, s));
    MXL_TRY(hipStreamSynchronize(s));
    if (h) {
        set_error(std::string(who) + ((h & 1) ? ": rowPtr does not rise from 0 to nnz" : ": column index out of range"));
        return MX_ERR_ARG;
    }
    return MX_OK;
}

hipError_t launch_lines_per_gather(mx_dtype dtype, int nnz, const int *col_dev, int most, unsigned long long *sum, long long *sampled, hipStream_t s)
{
    using namespace mxl;
    const long long windows = nnz / 64, stride = std::max<long long>(1, windows / most);
    *sampled = windows / stride;
    if (*sampled <= 0) return hipSuccess;
    hipLaunchKernelGGL(window_lines_kernel, dim3((unsigned)std::min<long long>(kLinesBlocks, (*sampled + 3) / 4)), dim3(kBlock), 0, s, col_dev, *sampled, stride, 64 / elem_size(dtype),
                       sum);
    return hipGetLastError();
}
int lines_per_gather_device(mx_dtype dtype, int nnz, const int *col_dev, hipStream_t s, double *out)
{
    using namespace mxl;
    *out = 1.0;
    if (nnz < 64) return MX_OK;
    Buf sum;
    MXL_TRY(mx::dev_malloc(&sum.p, 256));
    MXL_TRY(hipMemsetAsync(sum.p, 0, 256, s));
    long long sampled = 0;
    MXL_TRY(launch_lines_per_gather(dtype, nnz, col_dev, 65536, sum.as<unsigned long long>(), &sampled, s));
    unsigned long long h = 0;
    MXL_TRY(hipMemcpyAsync(&h, sum.p, 8, hipMemcpyDeviceToHost, s));
    MXL_TRY(hipStreamSynchronize(s));
    *out = (double)h / (double)sampled;
    return MX_OK;
}

// The row-tile form (DeviceCsr) of a CSR matrix in device memory: what upload_csr makes from host
// arrays.  `desc` = the workgroups' row ranges (pack_rows, made on the host from the row pointers).
int upload_csr_device(mx_dtype dtype, int rows, int cols, int nnz, const int *rowPtr_dev, const int *col_dev, const void *val_dev,
                      const std::vector<int> &desc, bool scan, DeviceCsr &A, hipStream_t s)
{
    using namespace mxl;
    const size_t es = (size_t)elem_size(dtype);
    A = DeviceCsr();
    A.rows = rows;
    A.cols = cols;
    A.nnz = nnz;
    A.npt = csr_entries_per_lane(dtype);
    A.scan = scan;
    A.nBlocks = (int)desc.size() / 4;
    MXL_TRY(mx::dev_malloc((void **)&A.rowPtr, ((size_t)rows + 1) * 4));
    MXL_TRY(hipMemcpyAsync(A.rowPtr, rowPtr_dev, ((size_t)rows + 1) * 4, hipMemcpyDeviceToDevice, s));
    MXL_TRY(mx::dev_malloc(&A.val, ((size_t)nnz + kCsrPad) * es));
    MXL_TRY(hipMemsetAsync((unsigned char *)A.val + (size_t)nnz * es, 0, (size_t)kCsrPad * es, s));
    if (nnz) MXL_TRY(hipMemcpyAsync(A.val, val_dev, (size_t)nnz * es, hipMemcpyDeviceToDevice, s));
    MXL_TRY(mx::dev_malloc((void **)&A.blockDesc, std::max<size_t>(desc.size(), 4) * 4));
    if (!desc.empty()) MXL_TRY(hipMemcpyAsync(A.blockDesc, desc.data(), desc.size() * 4, hipMemcpyHostToDevice, s));
    bool narrow = mx::opt().csr_col16 && nnz > 0;
    Buf lo, wide;
    if (narrow) {
        MXL_TRY(mx::dev_malloc(&lo.p, std::max<size_t>((size_t)A.nBlocks, 1) * 4));
        MXL_TRY(mx::dev_malloc(&wide.p, 256));
        MXL_TRY(hipMemsetAsync(wide.p, 0, 256, s));
        hipLaunchKernelGGL(block_ranges_kernel, grid((long long)A.nBlocks * 64), dim3(kBlock), 0, s, (const int4 *)A.blockDesc, col_dev,
                           A.nBlocks, lo.as<int>(), wide.as<int>());
        MXL_TRY(hipGetLastError());
        int w = 0;
        MXL_TRY(hipMemcpyAsync(&w, wide.p, 4, hipMemcpyDeviceToHost, s));
        MXL_TRY(hipStreamSynchronize(s));
        narrow = w == 0;
    }
    if (narrow) {
        MXL_TRY(mx::dev_malloc((void **)&A.col16, ((size_t)nnz + kCsrPad) * 2));
        MXL_TRY(hipMemsetAsync(A.col16 + nnz, 0, (size_t)kCsrPad * 2, s));
        hipLaunchKernelGGL(narrow_columns_kernel, grid((long long)A.nBlocks * 64), dim3(kBlock), 0, s, (const int4 *)A.blockDesc, col_dev,
                           (const int *)lo.p, A.nBlocks, A.col16);
        MXL_TRY(hipGetLastError());
        A.colBase = (int *)lo.take();
        if (nnz >= 65536 && mx::opt().csr_dict != 0) {
            Buf codes;
            std::vector<unsigned char> dict;
            int nd = 0, rc;
            if (dtype == MX_F64) rc = device_value_dict<double>((const double *)val_dev, nnz, codes, dict, &nd, s, 256, kCsrPad);
            else rc = device_value_dict<_Float16>((const _Float16 *)val_dev, nnz, codes, dict, &nd, s, 256, kCsrPad);
            if (rc) return rc;
            if (nd > 0) {
                A.codes = (unsigned char *)codes.take();
                MXL_TRY(mx::dev_malloc(&A.dict, dict.size()));
                MXL_TRY(hipMemcpyAsync(A.dict, dict.data(), dict.size(), hipMemcpyHostToDevice, s));
                MXL_TRY(hipStreamSynchronize(s));
                A.nDict = nd;
            }
        }
    } else {
        MXL_TRY(mx::dev_malloc((void **)&A.col, ((size_t)nnz + kCsrPad) * 4));
        MXL_TRY(hipMemsetAsync(A.col + nnz, 0, (size_t)kCsrPad * 4, s));
        if (nnz) MXL_TRY(hipMemcpyAsync(A.col, col_dev, (size_t)nnz * 4, hipMemcpyDeviceToDevice, s));
    }
    MXL_TRY(hipStreamSynchronize(s));
    return MX_OK;
}

int build_slices_device(mx_dtype dtype, int rows, int cols, int nnz, const int *rowPtr_dev, const int *col_dev, const void *val_dev,
                        int nCU, int S, const char *elsewhere_dev, DeviceSlices &D, hipStream_t s, std::vector<int> *segPtrOut,
                        std::vector<int> *segIdxOut, int fused)
{
    if (rows < 1 || cols < 1 || nnz < 0 || S < 1 || !rowPtr_dev || (nnz > 0 && (!col_dev || !val_dev))) {
        set_error("slice layout on the device: bad argument");
        return MX_ERR_ARG;
    }
    MXL_TRY(prepare_slice_kernels(dtype));
    if (dtype == MX_F64)
        return build_slices_device_t<double>(dtype, rows, cols, nnz, rowPtr_dev, col_dev, (const double *)val_dev, nCU, S, elsewhere_dev, D,
                                             s, segPtrOut, segIdxOut, fused);
    return build_slices_device_t<_Float16>(dtype, rows, cols, nnz, rowPtr_dev, col_dev, (const _Float16 *)val_dev, nCU, S, elsewhere_dev,
                                           D, s, segPtrOut, segIdxOut, fused);
}

}  // namespace mx

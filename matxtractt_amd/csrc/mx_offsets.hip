// The CSR part of a matrix whose rows repeat a pattern of column offsets -- a stencil on a
// structured grid with constant or variable coefficients, a banded operator with a few diagonals.
// Chunks of consecutive rows share one list of offsets (column - row, ascending), so a column costs
// nothing per entry and x is read in contiguous stretches instead of gathered.  The reference reads
// a column id per entry whatever the matrix (src/spmv_kernel/cdSpMV.cu:244-392).
//
// This file has the kernel, its launcher, and the routine that finds out on the device whether a
// matrix is of this kind and lays it out.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdint>
#include <cstring>
#include <string>
#include <vector>

#include <rocprim/device/device_scan.hpp>

#include "mx_device.h"
#include "mx_internal.h"

namespace mxo {

typedef int v4i32 __attribute__((ext_vector_type(4)));
typedef int v2i32 __attribute__((ext_vector_type(2)));

constexpr int kBlock = 256;
static_assert(kBlock == 4 * 64, "mx::offsets_blocks counts workgroups of four waves");
constexpr int kMaxOffsets = mx::kOffsetsMost;  // most distinct offsets of a chunk
constexpr int kTable = 2 * kMaxOffsets;        // slots of the table the offsets of a chunk are collected in
constexpr int kFree = (int)0x80000000;         // no offset: columns and rows are not negative

template <typename VT, bool DICT>
struct Form {
    static constexpr int R = sizeof(VT) == 8 ? 2 : 4;                              // consecutive rows of a lane
    static constexpr int kUnitBytes = mx::offsets_unit_bytes(DICT);                // what a lane loads at a time
    static constexpr int U = kUnitBytes / (R * (DICT ? 1 : (int)sizeof(VT)));      // offsets those bytes cover
    static constexpr int kRows = 64 * R;                                           // rows of a chunk
    static_assert(kRows == mx::offsets_chunk_rows(sizeof(VT) == 8), "the host looks at chunks of as many rows");
    typedef VT XV __attribute__((ext_vector_type(R), aligned(sizeof(VT))));        // R consecutive x, at any element
    typedef typename std::conditional<DICT, v2i32, v4i32>::type Unit;
    typedef typename std::conditional<sizeof(VT) == 8, double, float>::type AT;
};

template <bool KEEP, typename T>
__device__ __forceinline__ T unit_load(const T *p)
{
    if constexpr (KEEP) return *p;
    else return __builtin_nontemporal_load(p);
}

// acc[i] += value * x for the R rows of a lane and the U offsets of one unit.
// A place of the layout that no entry of the matrix owns (an offset that other rows of the chunk have
// and this one has not) holds -0.0, or code 255: its x is not used, whatever it is -- a row's sum must
// not become NaN because a neighbour's x is infinite.  (A matrix that stores such a value itself does
// not take this form; -0.0 stands for every binary64 with the upper half 0x80000000 here.)
template <typename VT, bool DICT>
__device__ __forceinline__ void unit_add(const typename Form<VT, DICT>::Unit &u, const VT (&xv)[Form<VT, DICT>::U][Form<VT, DICT>::R],
                                         typename Form<VT, DICT>::AT (&acc)[Form<VT, DICT>::R],
                                         const typename Form<VT, DICT>::AT *dict)
{
    typedef Form<VT, DICT> F;
    typedef typename F::AT AT;
#pragma unroll
    for (int j = 0; j < F::U; ++j)
#pragma unroll
        for (int i = 0; i < F::R; ++i) {
            const int e = j * F::R + i;  // place inside the unit
            if constexpr (DICT) {
                const int code = (int)(((unsigned)u[e >> 2] >> (8 * (e & 3))) & 255u);
                acc[i] += dict[code] * (code == 255 ? (AT)0 : (AT)xv[j][i]);
            } else if constexpr (sizeof(VT) == 8) {
                const int lo = u[2 * e], hi = u[2 * e + 1];
                const double v = __builtin_bit_cast(double, ((unsigned long long)(unsigned)hi << 32) | (unsigned)lo);
                acc[i] += v * (hi == (int)0x80000000 ? 0.0 : xv[j][i]);
            } else {
                const unsigned h = ((unsigned)u[e >> 1] >> (16 * (e & 1))) & 0xffffu;
                const float v = (float)__builtin_bit_cast(_Float16, (unsigned short)h);
                acc[i] += v * (h == 0x8000u ? 0.0f : (float)xv[j][i]);
            }
        }
}

// A chunk is 64 * R consecutive rows, R of them per lane, and W waves share one: each takes a contiguous
// part of its units, and with W > 1 the parts are added up through LDS in the order of the waves.  Per unit
// (16 bytes of values per lane, 8 bytes of codes) a lane reads its values -- the wave one contiguous
// stretch -- and for each of the unit's offsets R consecutive x, again contiguous across the wave; the
// offsets are the same for all lanes (scalar loads).  No column ids, no cross-lane traffic; y is written
// once, in order.  What bounds it is the stream of values (275.9 MB a product in 48.3 us, 5.7 TB/s; 17.4 MB that stay
// in the caches in 6.0), or on small matrices the trips to memory of a wave: a round takes eight offsets' worth (four at the end if that is enough), all of its loads ahead of its
// sums; a place beyond the wave's last unit reads that unit again and counts as "no entry".
// A chunk whose offsets reach outside x for some row (flag 1) or past the last row (flag 2) takes the
// form with every column clamped.
// Measured against the forms these matrices had before, three plans in turn (us): 27 points, 18.9 million binary64
// entries of their own value 28.6, row tiles 47.0; 26.5 million with two values 13.7, slices with one byte per value
// 35.7; 31.6 million binary16 12.7, slices 38.3; 56 thousand binary64 3.3, row tiles 3.3.
template <typename VT, bool DICT, bool KEEP, int W>
__global__ __launch_bounds__(kBlock) void csr_offsets_kernel(const int4 *__restrict__ chunk, const int *__restrict__ offs,
                                                             const void *__restrict__ stream, const VT *__restrict__ dictG,
                                                             const VT *__restrict__ x, VT *__restrict__ y, int rows, int cols,
                                                             int nChunks)
{
    typedef Form<VT, DICT> F;
    typedef typename F::AT AT;
    typedef typename F::Unit Unit;
    constexpr int R = F::R, U = F::U, WAVES = kBlock / 64;
    __shared__ AT dictL[DICT ? 256 : 1];
    __shared__ AT part[W > 1 ? WAVES : 1][W > 1 ? 64 * R : 1];
    if constexpr (DICT) {
        dictL[threadIdx.x] = (AT)dictG[threadIdx.x];
        __syncthreads();
    }
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6)), w = wave % W;
    // every XCD walks one contiguous range of chunks: the x of neighbouring chunks lives in one L2
    const int q = gridDim.x >> 3, rem = gridDim.x & 7, xcd = blockIdx.x & 7;
    const int block = xcd * q + min(xcd, rem) + (int)(blockIdx.x >> 3);
    const int c = block * (WAVES / W) + wave / W;
    const bool live = c < nChunks;
    const int4 d = chunk[live ? c : nChunks - 1];
    const int all = __builtin_amdgcn_readfirstlane(d.z), flags = __builtin_amdgcn_readfirstlane(d.w), share = (all + W - 1) / W;
    const int u0 = min(w * share, all), nUnits = live ? min(share, all - u0) : 0;  // this wave's part
    // (a scalar base and a 32-bit offset per lane: the address of a load costs no vector registers)
    const unsigned char *su = (const unsigned char *)stream + ((size_t)__builtin_amdgcn_readfirstlane(d.x) + u0) * (64 * F::kUnitBytes);
    const int *of = offs + __builtin_amdgcn_readfirstlane(d.y) + u0 * U;
    const unsigned suLane = (unsigned)lane * F::kUnitBytes, xLane = (unsigned)lane * (R * (unsigned)sizeof(VT));
    const int r0 = c * F::kRows + R * lane;
    AT acc[R];
#pragma unroll
    for (int i = 0; i < R; ++i) acc[i] = 0;
    if (flags == 0) {
        const VT *xc = x + (size_t)c * F::kRows;
        auto round = [&](int u, auto n, auto masked) {  // `n` units from u on
            constexpr int N = decltype(n)::value;
            constexpr bool MASK = decltype(masked)::value;
            Unit v[N];
            VT xv[N][U][R];
#pragma unroll
            for (int k = 0; k < N; ++k) {
                const int at = MASK ? min(u + k, nUnits - 1) : u + k;
                v[k] = unit_load<KEEP>((const Unit *)(su + (size_t)at * (64 * F::kUnitBytes) + suLane));
            }
#pragma unroll
            for (int k = 0; k < N; ++k)
#pragma unroll
                for (int j = 0; j < U; ++j) {
                    const int at = MASK ? min(u + k, nUnits - 1) : u + k;
                    const typename F::XV t = *(const typename F::XV *)((const unsigned char *)(xc + of[at * U + j]) + xLane);
#pragma unroll
                    for (int i = 0; i < R; ++i) xv[k][j][i] = t[i];
                }
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int k = 0; k < N; ++k) {
                if (MASK && u + k >= nUnits) {
#pragma unroll
                    for (int i = 0; i < F::kUnitBytes / 4; ++i) v[k][i] = DICT ? -1 : sizeof(VT) == 8 ? (int)0x80000000 : (int)0x80008000;
                }
                unit_add<VT, DICT>(v[k], xv[k], acc, dictL);
            }
        };
        constexpr int N = 8 / U;
        int u = 0;
        for (; u + N <= nUnits; u += N) round(u, std::integral_constant<int, N>(), std::false_type());
        if (u < nUnits) {
            if (N > 1 && nUnits - u <= N / 2) round(u, std::integral_constant<int, (N > 1 ? N / 2 : 1)>(), std::true_type());
            else round(u, std::integral_constant<int, N>(), std::true_type());
        }
    } else {
        for (int u = 0; u < nUnits; ++u) {
            const Unit v = unit_load<KEEP>((const Unit *)(su + (size_t)u * (64 * F::kUnitBytes) + suLane));
            VT xv[U][R];
#pragma unroll
            for (int j = 0; j < U; ++j) {
                const long long off = of[u * U + j];
#pragma unroll
                for (int i = 0; i < R; ++i) xv[j][i] = x[min(max((long long)r0 + i + off, 0ll), (long long)cols - 1)];
            }
            unit_add<VT, DICT>(v, xv, acc, dictL);
        }
    }
    if constexpr (W > 1) {
#pragma unroll
        for (int i = 0; i < R; ++i) part[wave][i * 64 + lane] = acc[i];
        __syncthreads();
        if (w != 0) return;
#pragma unroll
        for (int k = 1; k < W; ++k)
#pragma unroll
            for (int i = 0; i < R; ++i) acc[i] += part[wave + k][i * 64 + lane];
    }
    if (!live) return;
    if (r0 + R <= rows) {
        typename F::XV t;
#pragma unroll
        for (int i = 0; i < R; ++i) t[i] = (VT)acc[i];
        *(typename F::XV *)(y + r0) = t;
    } else {
#pragma unroll
        for (int i = 0; i < R; ++i)
            if (r0 + i < rows) y[r0 + i] = (VT)acc[i];
    }
}

// ---- laying a matrix out ----------------------------------------------------------------------------------

// The distinct offsets of every chunk (one workgroup each), ascending, into offs[chunk][kMaxOffsets] and their
// number into count[chunk].  totals[0] = 1 as soon as a chunk has more than kMaxOffsets; the workgroups that
// start after that leave at once.  A workgroup takes the chunk's entries as they lie, so a matrix of another kind is left after its first
// few of them.  (A wave to a chunk with a row to a lane walked the rows one entry at a time: 190 us for 700 thousand rows of a power law, so 19; a stencil of 290 thousand rows 33 and 31.)
__global__ __launch_bounds__(kBlock) void offset_lists_kernel(const int *__restrict__ rowPtr, const int *__restrict__ col, int rows,
                                                              int chunkRows, int *__restrict__ offs, int *__restrict__ count,
                                                              int *totals)
{
    __shared__ int start[mx::offsets_chunk_rows(false) + 1];
    __shared__ int table[kTable];
    __shared__ int list[kMaxOffsets];
    __shared__ int found, n, stop;
    const int c = blockIdx.x, tid = threadIdx.x;
    const int r0 = c * chunkRows, inside = min(chunkRows, rows - r0);
    if (tid == 0) {
        stop = *(volatile int *)totals;  // (looked at once: all threads go or all stay)
        found = n = 0;
    }
    for (int i = tid; i <= inside; i += kBlock) start[i] = rowPtr[r0 + i];
    for (int i = tid; i < kTable; i += kBlock) table[i] = kFree;
    __syncthreads();
    if (stop) return;
    bool tooMany = false;
    for (int p = start[0] + tid; p < start[inside] && !tooMany; p += kBlock) {
        int r = 0;  // the last row that begins at or before p
#pragma unroll
        for (int half = mx::offsets_chunk_rows(false) / 2; half; half >>= 1)
            if (r + half < inside && start[r + half] <= p) r += half;
        const int off = col[p] - (r0 + r);
        unsigned h = ((unsigned)off * 2654435761u) >> 25;  // the upper seven bits
        static_assert(kTable == 128, "seven bits of the product number the slots");
        bool placed = false;
        for (int step = 0; step < kTable && !placed && !tooMany; ++step) {
            int t = *(volatile int *)&table[h];
            if (t == kFree) {
                if (*(volatile int *)&found > kMaxOffsets) {
                    tooMany = true;
                } else {
                    t = atomicCAS(&table[h], kFree, off);
                    if (t == kFree) {
                        atomicAdd(&found, 1);
                        placed = true;
                    }
                }
            }
            if (t == off) placed = true;
            h = (h + 1) & (kTable - 1);
            if (!placed && *(volatile int *)&found > kMaxOffsets) tooMany = true;
        }
        tooMany = tooMany || !placed || *(volatile int *)&found > kMaxOffsets;
    }
    __syncthreads();
    // (others may have passed the test above together: the count decides.  A table that is full before it has been counted past
    // kMaxOffsets holds more than that, too)
    if (__syncthreads_or(tooMany) || found > kMaxOffsets) {
        if (tid == 0 && *(volatile int *)totals == 0) *(volatile int *)totals = 1;  // (stores to one word take turns)
        return;
    }
    for (int i = tid; i < kTable; i += kBlock) {
        const int t = table[i];
        if (t != kFree) list[atomicAdd(&n, 1)] = t;
    }
    __syncthreads();
    if (tid < n) {
        const int v = list[tid];
        int rank = 0;
        for (int k = 0; k < n; ++k) rank += list[k] < v;
        offs[(size_t)c * kMaxOffsets + rank] = v;
    }
    if (tid == 0) count[c] = n;
}

// units[c] = units of chunk c (one more element, zero); totals[1] += units, totals[2] = most offsets of a chunk
__global__ __launch_bounds__(kBlock) void chunk_units_kernel(const int *__restrict__ count, int nChunks, int U, int *__restrict__ units,
                                                             int *__restrict__ totals)
{
    const int c = blockIdx.x * kBlock + threadIdx.x;
    const int n = c < nChunks && !totals[0] ? (count[c] + U - 1) / U : 0;
    if (c <= nChunks) units[c] = n;
    int sum = n;
    for (int o = 32; o > 0; o >>= 1) sum += __shfl_xor(sum, o);
    int most = c < nChunks && !totals[0] ? count[c] : 0;
    for (int o = 32; o > 0; o >>= 1) most = max(most, __shfl_xor(most, o));
    if ((threadIdx.x & 63) == 0 && sum) {
        atomicAdd(totals + 1, sum);
        atomicMax(totals + 2, most);
    }
}

// The descriptor, the final offsets (the last one repeated up to whole units) and the values of one chunk per
// workgroup: the entries are taken as they lie, their values are put together in LDS and leave in one contiguous stretch.
// bad |= 1: a row names a column twice (two entries want one place: fewer places are taken than there are entries); bad |= 2:
// an entry holds what stands for "no entry".  (With a row to a thread, which walked it: 135 us for 7.6 million binary64 entries; so 46.)
template <typename VT, bool DICT>
__global__ __launch_bounds__(kBlock) void chunk_values_kernel(const int *__restrict__ rowPtr, const int *__restrict__ col,
                                                              const VT *__restrict__ val, const unsigned char *__restrict__ code,
                                                              const int *__restrict__ offsIn, const int *__restrict__ count,
                                                              const int *__restrict__ unit0, int rows, int cols, int4 *__restrict__ chunk,
                                                              int *__restrict__ offs, void *__restrict__ stream, int *__restrict__ bad)
{
    typedef Form<VT, DICT> F;
    typedef typename std::conditional<DICT, unsigned char, typename std::conditional<sizeof(VT) == 8, unsigned long long, unsigned short>::type>::type S;
    constexpr int R = F::R, U = F::U, PU = R * U;  // places of a lane's unit
    extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
    __shared__ int list[kMaxOffsets], start[F::kRows + 1];
    S *tile = (S *)smem;  // [units][64 lanes][PU]
    const int c = blockIdx.x, tid = threadIdx.x, n = count[c], nUnits = (n + U - 1) / U, u0 = unit0[c];
    const int r0 = c * F::kRows, r1 = min(r0 + F::kRows, rows);
    if (tid < kMaxOffsets) list[tid] = offsIn[(size_t)c * kMaxOffsets + max(min(tid, n - 1), 0)];
    S none;
    if constexpr (DICT) none = 255;
    else none = (S)((S)1 << (8 * sizeof(S) - 1));
    for (int i = tid; i <= r1 - r0; i += kBlock) start[i] = rowPtr[r0 + i];
    for (int i = tid; i < nUnits * 64 * PU; i += kBlock) tile[i] = none;
    __syncthreads();
    for (int i = tid; i < nUnits * U; i += kBlock) offs[(size_t)u0 * U + i] = list[min(i, n - 1)];
    if (tid == 0) {
        int flags = 0;
        if (n > 0 && (r0 + list[0] < 0 || (long long)r0 + F::kRows - 1 + list[n - 1] >= cols)) flags |= 1;
        if (r0 + F::kRows > rows) flags |= 2;
        chunk[c] = int4{u0, u0 * U, nUnits, flags};
    }
    int wrong = 0;
    const int p0 = start[0], size = start[r1 - r0] - p0;
    constexpr int AHEAD = 4;  // entries of a thread on their way at a time
    for (int i0 = tid; i0 < size; i0 = mx::next_of(i0, size, AHEAD * kBlock)) {
        int ci[AHEAD];
        S vi[AHEAD];
#pragma unroll
        for (int k = 0; k < AHEAD; ++k) {
            const int p = p0 + min(mx::next_of(i0, size, k * kBlock), size - 1);
            ci[k] = col[p];
            if constexpr (DICT) vi[k] = code[p];
            else vi[k] = __builtin_bit_cast(S, val[p]);
        }
#pragma unroll
        for (int k = 0; k < AHEAD; ++k) {
            const int i = mx::next_of(i0, size, k * kBlock);
            if (i >= size) break;
            int r = 0;  // the last row that begins at or before the entry
#pragma unroll
            for (int half = F::kRows / 2; half; half >>= 1)
                if (r + half < r1 - r0 && start[r + half] - p0 <= i) r += half;
            const int off = ci[k] - (r0 + r);
            int lo = 0, hi = n - 1;
            while (lo < hi) {
                const int mid = (lo + hi) >> 1;
                if (list[mid] < off) lo = mid + 1;
                else hi = mid;
            }
            const S v = vi[k];
            if constexpr (!DICT) {
                if constexpr (sizeof(VT) == 8) wrong |= (unsigned)(v >> 32) == 0x80000000u ? 2 : 0;
                else wrong |= v == 0x8000u ? 2 : 0;
            }
            tile[((size_t)(lo / U) * 64 + r / R) * PU + (lo % U) * R + r % R] = v;
        }
    }
    __syncthreads();
    int taken = 0;
    for (int i = tid; i < nUnits * 64 * PU; i += kBlock) taken += tile[i] != none;
    for (int o = 32; o > 0; o >>= 1) taken += __shfl_xor(taken, o);
    if (tid == 0) list[0] = 0;  // (the list has been used)
    __syncthreads();
    if ((tid & 63) == 0) atomicAdd(&list[0], taken);
    __syncthreads();
    if (tid == 0 && list[0] != size) wrong |= 1;
    if (wrong) atomicOr(bad, wrong);
    const v2i32 *src = (const v2i32 *)smem;
    v2i32 *dst = (v2i32 *)((unsigned char *)stream + (size_t)u0 * 64 * F::kUnitBytes);
    for (int i = tid; i < nUnits * 64 * F::kUnitBytes / 8; i += kBlock) dst[i] = src[i];
}

struct Buf {
    void *p = nullptr;
    Buf() = default;
    Buf(const Buf &) = delete;
    Buf &operator=(const Buf &) = delete;
    ~Buf()
    {
        if (p) (void)mx::dev_free(p);
    }
};
inline dim3 grid(long long n) { return dim3((unsigned)((std::max<long long>(n, 1) + kBlock - 1) / kBlock)); }

}  // namespace mxo

#define MXO_TRY(call)                                                                                     \
    do {                                                                                                  \
        hipError_t e_ = (call);                                                                           \
        if (e_ != hipSuccess) {                                                                           \
            mx::set_error(std::string("offset layout on the device: ") + #call + ": " + hipGetErrorString(e_)); \
            return e_ == hipErrorOutOfMemory ? MX_ERR_ALLOC : MX_ERR_DEVICE;                              \
        }                                                                                                 \
    } while (0)

namespace mx {

template <typename VT, bool DICT>
static int offsets_values(const int *rowPtr, const int *col, const VT *val, const unsigned char *code, const int *lists, const int *count,
                          const int *unit0, int most, DeviceOffsets &D, int *bad, hipStream_t s)
{
    using namespace mxo;
    typedef Form<VT, DICT> F;
    const size_t lds = (size_t)((most + F::U - 1) / F::U) * 64 * F::kUnitBytes;
    if (lds > 65536) MXO_TRY(hipFuncSetAttribute((const void *)chunk_values_kernel<VT, DICT>, hipFuncAttributeMaxDynamicSharedMemorySize, 163840 - 1024));
    hipLaunchKernelGGL((chunk_values_kernel<VT, DICT>), dim3(D.nChunks), dim3(kBlock), lds, s, rowPtr, col, val, code, lists, count, unit0, D.rows,
                       D.cols, (int4 *)D.chunk, D.offs, D.stream, bad);
    MXO_TRY(hipGetLastError());
    return MX_OK;
}

int build_offsets_device(mx_dtype dtype, int rows, int cols, int nnz, const int *rowPtr_dev, const int *col_dev, const void *val_dev,
                         DeviceOffsets &D, hipStream_t s)
{
    using namespace mxo;
    D = DeviceOffsets();
    // (what cannot pass is not looked at: too few rows to fill a chunk, more entries a row than a chunk has offsets)
    if (!offsets_size_ok(rows, cols, nnz)) return MX_OK;
    const int R = dtype == MX_F64 ? 2 : 4, chunkRows = 64 * R, nChunks = (rows + chunkRows - 1) / chunkRows;
    Buf lists, count, units, unit0, totals, tmp;
    size_t scanBytes = 0;
    MXO_TRY(rocprim::exclusive_scan(nullptr, scanBytes, (const int *)nullptr, (int *)nullptr, 0, (size_t)nChunks + 1, rocprim::plus<int>(), s));
    MXO_TRY(mx::dev_malloc(&lists.p, (size_t)nChunks * kMaxOffsets * 4));
    MXO_TRY(mx::dev_malloc(&count.p, ((size_t)nChunks + 1) * 4));
    MXO_TRY(mx::dev_malloc(&units.p, ((size_t)nChunks + 1) * 4));
    MXO_TRY(mx::dev_malloc(&unit0.p, ((size_t)nChunks + 1) * 4));
    MXO_TRY(mx::dev_malloc(&totals.p, 256));
    MXO_TRY(mx::dev_malloc(&tmp.p, scanBytes + 256));
    MXO_TRY(hipMemsetAsync(totals.p, 0, 256, s));
    int *tot = (int *)totals.p;
    hipLaunchKernelGGL(offset_lists_kernel, dim3(nChunks), dim3(kBlock), 0, s, rowPtr_dev, col_dev, rows, chunkRows, (int *)lists.p, (int *)count.p, tot);
    // (with whole 16-byte units of values; a dictionary counts again below)
    int U = 16 / (R * elem_size(dtype));
    hipLaunchKernelGGL(chunk_units_kernel, grid((long long)nChunks + 1), dim3(kBlock), 0, s, (const int *)count.p, nChunks, U, (int *)units.p, tot);
    MXO_TRY(hipGetLastError());
    int h[3] = {0, 0, 0};
    MXO_TRY(hipMemcpyAsync(h, totals.p, sizeof(h), hipMemcpyDeviceToHost, s));
    MXO_TRY(hipStreamSynchronize(s));
    if (h[0] || h[1] <= 0) return MX_OK;
    const long long places = (long long)h[1] * U * chunkRows;
    if ((double)places > kOffsetsFill * (double)nnz + 64.0 * chunkRows || places / (U * R) > 2000000000LL) return MX_OK;

    // ---- the matrix is of this kind: values, or one byte per value where there are at most 255 of them
    D.rows = rows;
    D.cols = cols;
    D.nnz = nnz;
    D.nChunks = nChunks;
    void *codes = nullptr;
    std::vector<unsigned char> dict;
    int rc = MX_OK;
    if (nnz >= 65536 && mx::opt().csr_dict != 0)
        if ((rc = value_dict_device(dtype, val_dev, nnz, 255, &codes, dict, &D.nDict, s))) return rc;
    Buf codesHold;
    codesHold.p = codes;
    if (!offsets_lists_pay(dtype == MX_F64, D.nDict > 0, h[2], nnz)) {
        D = DeviceOffsets();
        return MX_OK;
    }
    int unitBytes = 16;
    if (D.nDict > 0) {
        unitBytes = offsets_unit_bytes(true);
        U = unitBytes / R;
        MXO_TRY(hipMemsetAsync(tot + 1, 0, 4, s));
        hipLaunchKernelGGL(chunk_units_kernel, grid((long long)nChunks + 1), dim3(kBlock), 0, s, (const int *)count.p, nChunks, U, (int *)units.p,
                           tot);
        MXO_TRY(hipGetLastError());
        MXO_TRY(hipMemcpyAsync(h, totals.p, sizeof(h), hipMemcpyDeviceToHost, s));
        MXO_TRY(hipStreamSynchronize(s));
    }
    D.units = h[1];
    D.unitBytes = unitBytes;
    D.nOffs = (long long)D.units * U;
    MXO_TRY(rocprim::exclusive_scan(tmp.p, scanBytes, (const int *)units.p, (int *)unit0.p, 0, (size_t)nChunks + 1, rocprim::plus<int>(), s));
    auto fail = [&](int code) {
        free_offsets(D);
        return code;
    };
    auto body = [&]() -> int {
        MXO_TRY(mx::dev_malloc((void **)&D.chunk, (size_t)nChunks * 16));
        MXO_TRY(mx::dev_malloc((void **)&D.offs, (size_t)D.nOffs * 4));
        MXO_TRY(mx::dev_malloc(&D.stream, (size_t)D.units * 64 * unitBytes));
        if (D.nDict > 0) {
            MXO_TRY(mx::dev_malloc(&D.dict, dict.size()));
            MXO_TRY(hipMemcpyAsync(D.dict, dict.data(), dict.size(), hipMemcpyHostToDevice, s));
        }
        int *bad = tot + 3;
        const int *L = (const int *)lists.p, *C = (const int *)count.p, *U0 = (const int *)unit0.p;
        const unsigned char *K = (const unsigned char *)codes;
        int r;
        if (dtype == MX_F64)
            r = D.nDict > 0 ? offsets_values<double, true>(rowPtr_dev, col_dev, (const double *)val_dev, K, L, C, U0, h[2], D, bad, s)
                            : offsets_values<double, false>(rowPtr_dev, col_dev, (const double *)val_dev, K, L, C, U0, h[2], D, bad, s);
        else
            r = D.nDict > 0 ? offsets_values<_Float16, true>(rowPtr_dev, col_dev, (const _Float16 *)val_dev, K, L, C, U0, h[2], D, bad, s)
                            : offsets_values<_Float16, false>(rowPtr_dev, col_dev, (const _Float16 *)val_dev, K, L, C, U0, h[2], D, bad, s);
        if (r) return r;
        int hb = 0;
        MXO_TRY(hipMemcpyAsync(&hb, bad, 4, hipMemcpyDeviceToHost, s));
        MXO_TRY(hipStreamSynchronize(s));
        if (hb) free_offsets(D);  // (a column named twice, or a stored -0.0: another form takes the matrix)
        return MX_OK;
    };
    if ((rc = body())) return fail(rc);
    return MX_OK;
}

// (W as offsets_waves gives it for D: the grid is made from the same rule)
template <typename VT, int W>
static hipError_t launch_offsets_t(const DeviceOffsets &D, const void *x, void *y, hipStream_t s)
{
    const int wgs = offsets_blocks(sizeof(VT) == 8, D);
#define MX_LAUNCH_OFFSETS(DICT, KEEP)                                                                                                    \
    hipLaunchKernelGGL((mxo::csr_offsets_kernel<VT, DICT, KEEP, W>), dim3(wgs), dim3(mxo::kBlock), 0, s, (const int4 *)D.chunk, D.offs,    \
                       (const void *)D.stream, (const VT *)D.dict, (const VT *)x, (VT *)y, D.rows, D.cols, D.nChunks)
    if (D.nDict > 0 && D.keep) MX_LAUNCH_OFFSETS(true, true);
    else if (D.nDict > 0) MX_LAUNCH_OFFSETS(true, false);
    else if (D.keep) MX_LAUNCH_OFFSETS(false, true);
    else MX_LAUNCH_OFFSETS(false, false);
#undef MX_LAUNCH_OFFSETS
    return hipGetLastError();
}
hipError_t launch_offsets(mx_dtype dtype, const DeviceOffsets &D, const void *x, void *y, hipStream_t s)
{
    if (D.nChunks <= 0) return hipSuccess;
    const int waves = offsets_waves(dtype == MX_F64, D.nDict > 0, D.nOffs, D.nChunks);
    if (dtype == MX_F16) return waves == 1 ? launch_offsets_t<_Float16, 1>(D, x, y, s) : launch_offsets_t<_Float16, 4>(D, x, y, s);
    if (waves == 1) return launch_offsets_t<double, 1>(D, x, y, s);
    return waves == 2 ? launch_offsets_t<double, 2>(D, x, y, s) : launch_offsets_t<double, 4>(D, x, y, s);
}

}  // namespace mx

// The CSR part of a matrix whose neighbouring rows reach into one stretch of x -- a mesh numbered for a small
// bandwidth, a band without a pattern.  A workgroup takes consecutive rows, puts the window of x that they reach
// into LDS and gathers from there; a row belongs to one lane, y is written once, in order, in one launch.  The reference gathers x
// from memory for every entry whatever the matrix (src/spmv_kernel/cdSpMV.cu:244-392).
//
// This file has the kernel, its launcher, and the routine that finds out on the device whether a
// matrix is of this kind and lays it out.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <climits>
#include <cstdint>
#include <cstring>
#include <string>
#include <vector>

#include <rocprim/device/device_scan.hpp>

#include "mx_device.h"
#include "mx_internal.h"

namespace mxw {

typedef int v4i32 __attribute__((ext_vector_type(4)));
typedef int v2i32 __attribute__((ext_vector_type(2)));
typedef double v2f64 __attribute__((ext_vector_type(2)));

constexpr int kU = mx::kWindowUnit;  // entries of a row that a lane loads at a time
constexpr int kBlock = 256;          // of the kernels that lay out

// What a lane loads at a time: four 16-bit places in the window and four values.  A unit of a wave is one contiguous stretch:
// binary16 16 bytes a lane; binary64 the places of all lanes, then the first two values of all, then the other two.
template <typename VT>
struct Unit;
template <>
struct Unit<_Float16> {
    v4i32 d;
    template <bool KEEP>
    __device__ __forceinline__ void load(const unsigned char *p, int lane)
    {
        const v4i32 *q = (const v4i32 *)p + lane;
        if constexpr (KEEP) d = *q;
        else d = __builtin_nontemporal_load(q);
    }
    __device__ __forceinline__ int place(int j) const { return (int)(((unsigned)d[j >> 1] >> (16 * (j & 1))) & 0xffffu); }
    __device__ __forceinline__ float value(int j) const
    {
        return (float)__builtin_bit_cast(_Float16, (unsigned short)((unsigned)d[2 + (j >> 1)] >> (16 * (j & 1))));
    }
};
template <>
struct Unit<double> {
    v2i32 c;
    v2f64 a, b;
    template <bool KEEP>
    __device__ __forceinline__ void load(const unsigned char *p, int lane)
    {
        const v2i32 *qc = (const v2i32 *)p + lane;
        const v2f64 *qa = (const v2f64 *)(p + 512) + lane, *qb = qa + 64;
        if constexpr (KEEP) {
            c = *qc;
            a = *qa;
            b = *qb;
        } else {
            c = __builtin_nontemporal_load(qc);
            a = __builtin_nontemporal_load(qa);
            b = __builtin_nontemporal_load(qb);
        }
    }
    __device__ __forceinline__ int place(int j) const { return (int)(((unsigned)c[j >> 1] >> (16 * (j & 1))) & 0xffffu); }
    __device__ __forceinline__ double value(int j) const { return j < 2 ? a[j] : b[j - 2]; }
};

// One chunk -- 64 consecutive rows, a row per lane -- to a wave, WAVES of them to a workgroup.  The wave's
// first NB units are asked for before the window is copied, so both trips to memory run side by side; after that each
// unit is followed by the request for the one NB further on (the last one again where there is none).  A place that no entry owns
// names the zero behind the window and has the value zero, so a row's sum never touches an x that the row does not name.
// The few entries outside the window ("far": a step is one of them per lane, column -1 for none) are gathered from memory,
// on their way while the window is copied.  A chunk with a row of more than kWindowFarSteps of them is taken apart from the others: a
// workgroup of its own gathers everything, one step of eight waves at a time (in its own place it kept its CU's address unit
// busy long after the other workgroups were done: the ends of a band of 250 thousand rows, binary16, 17.0 us where the rest took 8.5).
// What bounds it is the stream of entries (250007 rows of 40 entries within 3000 of the diagonal, binary16: 40 MB in 9.8 us with what it
// takes to launch; binary64: 100 MB in 19.5).  Eight waves to a workgroup: with four a window is read twice as often (10.3 us); a chunk to
// a wave, because a chunk's units are then all on their way at once.
// Measured against what these matrices had before (us, column slices unless noted): binary16, 70 thousand rows of 40 within 3000
// 4.2, 8.2; 250 thousand 9.8, 13.2; 160 thousand of 25 within 6000 5.0, 10.0; 600 thousand of 16 within 1000 10.7, 14.3; 45
// thousand of 20 within 500 3.6, 5.1 (row tiles); a million of 8 within 200 13.0, 13.8 (row tiles); binary64, 70 thousand of 40 6.5, 11.4; 250
// thousand 19.5, 23.0; 600 thousand of 16 19.1, 24.2.
template <typename VT, bool KEEP, int WAVES>
__global__ __launch_bounds__(64 * WAVES) void csr_window_kernel(const int2 *__restrict__ window, const int4 *__restrict__ chunk,
                                                                const unsigned char *__restrict__ stream, const int *__restrict__ farCol,
                                                                const VT *__restrict__ farVal, const int *__restrict__ apart, const VT *__restrict__ x,
                                                                VT *__restrict__ y, int rows, int cols, int nChunks, int nApart, int zeroPlace)
{
    typedef typename std::conditional<sizeof(VT) == 8, double, float>::type AT;
    constexpr int EPV = 16 / (int)sizeof(VT), THREADS = 64 * WAVES, NB = sizeof(VT) == 8 ? 6 : 10, XR = 4, NF = mx::kWindowFarSteps;
    constexpr int UB = mx::window_unit_bytes(sizeof(VT) == 8);
    typedef VT XV __attribute__((ext_vector_type(EPV), aligned(sizeof(VT))));
    typedef VT LV __attribute__((ext_vector_type(EPV)));
    extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
    VT *xs = (VT *)smem;
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    if ((int)blockIdx.x < nApart) {
        // a chunk apart: all of its entries are gathered from memory, the waves share its steps
        const int c = apart[blockIdx.x];
        const int4 d = chunk[c];
        const int nf = __builtin_amdgcn_readfirstlane(d.w), share = (nf + WAVES - 1) / WAVES, k1 = min((wave + 1) * share, nf);
        const int *fc = farCol + (size_t)__builtin_amdgcn_readfirstlane(d.z) * 64 + lane;
        const VT *fv = farVal + (size_t)__builtin_amdgcn_readfirstlane(d.z) * 64 + lane;
        AT acc = 0;
        for (int k = wave * share; k < k1; k += 8) {
            int col[8];
            VT v[8], g[8];
#pragma unroll
            for (int j = 0; j < 8; ++j) {
                col[j] = fc[min(k + j, k1 - 1) * 64];
                v[j] = fv[min(k + j, k1 - 1) * 64];
            }
#pragma unroll
            for (int j = 0; j < 8; ++j) g[j] = x[max(col[j], 0)];
#pragma unroll
            for (int j = 0; j < 8; ++j)
                if (k + j < k1 && col[j] >= 0) acc += (AT)v[j] * (AT)g[j];
        }
        AT *part = (AT *)smem;
        part[tid] = acc;
        __syncthreads();
        if (wave > 0) return;
#pragma unroll
        for (int k = 1; k < WAVES; ++k) acc += part[k * 64 + lane];
        const int r = c * 64 + lane;
        if (r < rows) y[r] = (VT)acc;
        return;
    }
    // every XCD walks one contiguous range of rows: the x of neighbouring windows lives in one L2
    const int nb = (int)gridDim.x - nApart, bid = (int)blockIdx.x - nApart, q = nb >> 3, rem = nb & 7, xcd = bid & 7;
    const int b = xcd * q + min(xcd, rem) + (bid >> 3);
    const int2 w = window[b];  // first element, vectors
    const int c = b * WAVES + wave;
    const int4 d = chunk[min(c, nChunks - 1)];  // first unit, units (-1: a chunk apart), first far step, far steps
    const int u0 = __builtin_amdgcn_readfirstlane(d.x), f0 = __builtin_amdgcn_readfirstlane(d.z);
    const int n = c < nChunks ? max(__builtin_amdgcn_readfirstlane(d.y), 0) : 0, nf = n > 0 || d.y == 0 ? __builtin_amdgcn_readfirstlane(d.w) : 0;
    // (every array has a unit and a step to spare behind the last: a chunk without any may read there)
    const unsigned char *su = stream + (size_t)u0 * UB;
    const int *fc = farCol + (size_t)f0 * 64 + lane;
    const VT *fv = farVal + (size_t)f0 * 64 + lane;
    const int last = max(n - 1, 0), lastFar = max(nf - 1, 0);
    const int lastStart = cols - EPV;  // (the last vector of x starts here at the latest)
    XV xv[XR];
#pragma unroll
    for (int k = 0; k < XR; ++k) xv[k] = *(const XV *)(x + min(w.x + min(tid + k * THREADS, w.y - 1) * EPV, lastStart));
    int farC[NF];
    VT farV[NF], farX[NF];
#pragma unroll
    for (int k = 0; k < NF; ++k) {
        farC[k] = fc[min(k, lastFar) * 64];
        farV[k] = fv[min(k, lastFar) * 64];
    }
    Unit<VT> buf[NB];
#pragma unroll
    for (int k = 0; k < NB; ++k) buf[k].template load<KEEP>(su + (size_t)min(k, last) * UB, lane);
#pragma unroll
    for (int k = 0; k < NF; ++k) farX[k] = x[max(farC[k], 0)];
    auto keep = [&](int i, const XV &v) {
        const int s = w.x + i * EPV;
        if (s <= lastStart) {
            *(LV *)(xs + i * EPV) = v;
        } else {
            const int to = lastStart - w.x;  // (not negative: a window starts at a vector of x that is whole)
#pragma unroll
            for (int e = 0; e < EPV; ++e) xs[to + e] = v[e];
        }
    };
#pragma unroll
    for (int k = 0; k < XR; ++k)
        if (tid + k * THREADS < w.y) keep(tid + k * THREADS, xv[k]);
    for (int i = tid + XR * THREADS; i < w.y; i += THREADS) keep(i, *(const XV *)(x + min(w.x + i * EPV, lastStart)));
    if (tid == 0) xs[zeroPlace] = (VT)0;
    __syncthreads();
    AT acc = 0;
    auto add = [&](const Unit<VT> &u) {
        VT g[kU];
#pragma unroll
        for (int j = 0; j < kU; ++j) g[j] = xs[u.place(j)];
#pragma unroll
        for (int j = 0; j < kU; ++j) acc += (AT)u.value(j) * (AT)g[j];
    };
    int t = 0;
    for (; t + NB < n; t += NB) {
#pragma unroll
        for (int k = 0; k < NB; ++k) {
            add(buf[k]);
            buf[k].template load<KEEP>(su + (size_t)min(t + NB + k, last) * UB, lane);
        }
    }
#pragma unroll
    for (int k = 0; k < NB; ++k)
        if (t + k < n) add(buf[k]);
#pragma unroll
    for (int k = 0; k < NF; ++k)
        if (k < nf && farC[k] >= 0) acc += (AT)farV[k] * (AT)farX[k];
    const int r = c * 64 + lane;
    if (c < nChunks && d.y >= 0 && r < rows) y[r] = (VT)acc;
}

// ---- laying a matrix out ----------------------------------------------------------------------------------

constexpr int kBuckets = mx::kWindowBuckets;

// totals[0] = 1 where a row has more than kWindowLongest entries: a matrix with a tail of long rows is not looked at any
// further (16 million entries in a million rows: 0.28 ms of counting columns).  Few workgroups, one store each: stores to
// one word take turns (a wave of every 64 rows storing for itself: 61 us for a million rows with four in a thousand too long; so 13).
constexpr int kRowsBlocks = 256;
__global__ __launch_bounds__(kBlock) void window_rows_kernel(const int *__restrict__ rowPtr, int rows, int *totals)
{
    bool tooLong = false;
#pragma unroll 8
    for (long long r = (long long)blockIdx.x * kBlock + threadIdx.x; r < rows; r += kRowsBlocks * kBlock)
        tooLong |= rowPtr[r + 1] - rowPtr[r] > mx::kWindowLongest;
    if (__syncthreads_or(tooLong) && threadIdx.x == 0) *(volatile int *)totals = 1;
}

// The window of a workgroup's rows: of its entries' columns, counted in buckets, the stretch of at most `widest` elements
// that holds the most, without the ends that cost more as a part of the window (their x) than as far entries.  Per chunk the
// units and far steps that makes.  totals[0] = 1 as soon as a workgroup has more than three quarters of its entries outside
// (workgroups that start after that leave at once); totals[1] += units, totals[2] += far steps, totals[3] = most
// vectors of a window, totals[4] += entries gathered from memory, totals[5] += chunks apart.
__global__ __launch_bounds__(kBlock) void window_find_kernel(const int *__restrict__ rowPtr, const int *__restrict__ col, int rows, int cols,
                                                             int nChunks, int waves, int epv, int widest, int2 *__restrict__ window,
                                                             int *__restrict__ units, int *__restrict__ farSteps, int *__restrict__ apart, int *totals)
{
    __shared__ int hist[kBuckets];
    __shared__ int part[kBlock];
    __shared__ int over, sumUnits, sumFar, inside;
    __shared__ unsigned long long best;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    constexpr int BT = kBuckets / kBlock;
    if (tid == 0) {
        over = *(volatile int *)totals;  // (looked at once: all threads go or all stay)
        sumUnits = sumFar = inside = 0;
        best = 0;
    }
    __syncthreads();
    if (over) return;
    const int size = mx::window_bucket(cols, epv), wide = max(widest / size, 1);
    const int c0 = blockIdx.x * waves, c1 = min(c0 + waves, nChunks);
    const int r0 = c0 * 64, r1 = min(c1 * 64, rows), p0 = rowPtr[r0], p1 = rowPtr[r1];
    for (int i = tid; i < kBuckets; i += kBlock) hist[i] = 0;
    __syncthreads();
    for (int p = p0 + tid; p < p1; p += kBlock) atomicAdd(&hist[col[p] / size], 1);
    __syncthreads();
    // running sums, then the best window of `wide` buckets (the first of equally good ones)
    int own[BT], sum = 0;
#pragma unroll
    for (int k = 0; k < BT; ++k) sum += own[k] = hist[tid * BT + k];
    part[tid] = sum;
    __syncthreads();
    for (int off = 1; off < kBlock; off <<= 1) {
        const int o = tid >= off ? part[tid - off] : 0;
        __syncthreads();
        part[tid] += o;
        __syncthreads();
    }
    int run = part[tid] - sum;
    __syncthreads();
#pragma unroll
    for (int k = 0; k < BT; ++k) hist[tid * BT + k] = run += own[k];
    __syncthreads();
    for (int i = tid; i < kBuckets; i += kBlock) {
        const int in = hist[min(i + wide, kBuckets) - 1] - (i ? hist[i - 1] : 0);
        if (in > 0) atomicMax(&best, ((unsigned long long)in << 32) | (unsigned)(kBuckets - i));
    }
    __syncthreads();
    // (all threads the same walk) ends with few entries: kWindowTrim bytes a far entry against the bucket's x
    int lo = best ? kBuckets - (int)(best & 0xffffffffu) : 0, hi = min(lo + wide, kBuckets) - 1;
    const int few = size * (16 / epv) / mx::kWindowTrim;
    while (lo < hi && hist[lo] - (lo ? hist[lo - 1] : 0) <= few) ++lo;
    while (hi > lo && hist[hi] - hist[hi - 1] <= few) --hi;
    const int first = min((long long)lo * size, (long long)(cols - epv) / epv * epv), behind = (int)min((long long)(hi + 1) * size, (long long)cols);
    const int vecs = max((behind - first + epv - 1) / epv, 1);
    const int outside = p1 - p0 - (hist[hi] - (lo ? hist[lo - 1] : 0));
    // (before a lane walks its row: a matrix of another kind is found out by its first workgroups)
    if (size > widest || mx::window_scattered(outside, p1 - p0)) {
        if (tid == 0) *(volatile int *)totals = 1;
        return;
    }
    for (int c = c0 + wave; c < c1; c += kBlock / 64) {
        const int r = c * 64 + lane;
        int near = 0, far = 0;
        if (r < rows)
            for (int p = rowPtr[r], e = rowPtr[r + 1]; p < e; ++p) (unsigned)(col[p] - first) < (unsigned)(vecs * epv) ? ++near : ++far;
        int n = (near + kU - 1) / kU, f = far, in = near;
        for (int o = 32; o > 0; o >>= 1) {
            n = max(n, __shfl_xor(n, o));
            f = max(f, __shfl_xor(f, o));
            in += __shfl_xor(in, o);
        }
        int longest = near + far;
        for (int o = 32; o > 0; o >>= 1) longest = max(longest, __shfl_xor(longest, o));
        if (lane == 0) {
            const bool alone = f > mx::kWindowFarSteps;
            if (alone) {
                n = 0;
                f = longest;
                in = 0;
            }
            units[c] = n;
            farSteps[c] = f;
            apart[c] = alone;
            atomicAdd(&sumUnits, n);
            atomicAdd(&sumFar, f);
            atomicAdd(&inside, in);
            if (alone) atomicAdd(totals + 5, 1);
        }
    }
    __syncthreads();
    if (tid == 0) {
        window[blockIdx.x] = int2{first, vecs};
        atomicAdd(totals + 4, p1 - p0 - inside);
        atomicAdd(totals + 1, sumUnits);
        atomicAdd(totals + 2, sumFar);
        atomicMax(totals + 3, vecs);
    }
}

// A chunk's descriptor, units and far steps, one wave each: a lane walks its own row.
template <typename VT>
__global__ __launch_bounds__(kBlock) void window_fill_kernel(const int *__restrict__ rowPtr, const int *__restrict__ col, const VT *__restrict__ val,
                                                             const int2 *__restrict__ window, const int *__restrict__ unit0,
                                                             const int *__restrict__ far0, const int *__restrict__ apart0, int rows, int nChunks, int waves, int zeroPlace,
                                                             int4 *__restrict__ chunk, unsigned char *__restrict__ stream,
                                                             int *__restrict__ farCol, VT *__restrict__ farVal, int *__restrict__ apart)
{
    constexpr int UB = mx::window_unit_bytes(sizeof(VT) == 8), EPV = 16 / (int)sizeof(VT);
    const int c = blockIdx.x * (kBlock / 64) + (threadIdx.x >> 6), lane = threadIdx.x & 63;
    if (c >= nChunks) return;
    const int r = c * 64 + lane, u0 = unit0[c], n = unit0[c + 1] - u0, f0 = far0[c], nf = far0[c + 1] - f0;
    const int2 w = window[c / waves];
    const bool alone = apart0[c + 1] > apart0[c];
    if (lane == 0) {
        chunk[c] = int4{u0, alone ? -1 : n, f0, nf};
        if (alone) apart[apart0[c]] = c;
    }
    int p = r < rows ? rowPtr[r] : 0, f = 0;
    const int p1 = r < rows ? rowPtr[r + 1] : 0;
    for (int u = 0; u < n; ++u) {
        unsigned place[kU];
        VT v[kU];
#pragma unroll
        for (int j = 0; j < kU; ++j) {
            place[j] = (unsigned)zeroPlace;
            v[j] = (VT)0;
            while (p < p1) {
                const int at = col[p] - w.x;
                const VT value = val[p++];
                if ((unsigned)at < (unsigned)(w.y * EPV)) {
                    place[j] = (unsigned)at;
                    v[j] = value;
                    break;
                }
                if (f < nf) {
                    farCol[(size_t)(f0 + f) * 64 + lane] = at + w.x;
                    farVal[(size_t)(f0 + f) * 64 + lane] = value;
                    ++f;
                }
            }
        }
        unsigned char *out = stream + (size_t)(u0 + u) * UB;
        const v2i32 pl = {(int)(place[0] | (place[1] << 16)), (int)(place[2] | (place[3] << 16))};
        if constexpr (sizeof(VT) == 2) {
            auto bits = [&](int j) { return (unsigned)__builtin_bit_cast(unsigned short, v[j]); };
            ((v4i32 *)out)[lane] = v4i32{pl[0], pl[1], (int)(bits(0) | (bits(1) << 16)), (int)(bits(2) | (bits(3) << 16))};
        } else {
            ((v2i32 *)out)[lane] = pl;
            ((v2f64 *)(out + 512))[lane] = v2f64{v[0], v[1]};
            ((v2f64 *)(out + 512))[64 + lane] = v2f64{v[2], v[3]};
        }
    }
    for (; p < p1; ++p)  // (what is left of a row lies outside the window)
        if (f < nf) {
            farCol[(size_t)(f0 + f) * 64 + lane] = col[p];
            farVal[(size_t)(f0 + f) * 64 + lane] = val[p];
            ++f;
        }
    for (; f < nf; ++f) {
        farCol[(size_t)(f0 + f) * 64 + lane] = -1;
        farVal[(size_t)(f0 + f) * 64 + lane] = (VT)0;
    }
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

}  // namespace mxw

#define MXW_TRY(call)                                                                                     \
    do {                                                                                                  \
        hipError_t e_ = (call);                                                                           \
        if (e_ != hipSuccess) {                                                                           \
            mx::set_error(std::string("window layout on the device: ") + #call + ": " + hipGetErrorString(e_)); \
            return e_ == hipErrorOutOfMemory ? MX_ERR_ALLOC : MX_ERR_DEVICE;                              \
        }                                                                                                 \
    } while (0)

namespace mx {

template <typename VT, bool KEEP, int WAVES>
static const void *window_kernel()
{
    return (const void *)mxw::csr_window_kernel<VT, KEEP, WAVES>;
}

int build_windows_device(mx_dtype dtype, int rows, int cols, int nnz, const int *rowPtr_dev, const int *col_dev, const void *val_dev,
                         DeviceWindows &D, hipStream_t s)
{
    using namespace mxw;
    D = DeviceWindows();
    const bool f64 = dtype == MX_F64;
    const int es = elem_size(dtype), epv = 16 / es;
    if (!window_size_ok(f64, rows, cols, nnz)) return MX_OK;
    const int nChunks = (rows + 63) / 64, waves = kWindowWaves, nWG = (nChunks + waves - 1) / waves;
    const int widest = window_widest(f64, nnz, nWG);
    Buf counts, unit0, far0, apart0, tmp;
    size_t scanBytes = 0;
    const size_t chunkB = ((size_t)nChunks + 1) * 4, countB = (chunkB + 255) & ~(size_t)255;
    MXW_TRY(rocprim::exclusive_scan(nullptr, scanBytes, (const int *)nullptr, (int *)nullptr, 0, (size_t)nChunks + 1, rocprim::plus<int>(), s));
    MXW_TRY(mx::dev_malloc(&counts.p, 256 + 3 * countB));  // (cleared together: 10 us for each of them apart)
    int *const tot = (int *)counts.p, *const units = (int *)((char *)counts.p + 256), *const farSteps = (int *)((char *)units + countB),
               *const alone = (int *)((char *)farSteps + countB);
    MXW_TRY(mx::dev_malloc(&unit0.p, chunkB));
    MXW_TRY(mx::dev_malloc(&far0.p, chunkB));
    MXW_TRY(mx::dev_malloc(&apart0.p, chunkB));
    MXW_TRY(mx::dev_malloc(&tmp.p, scanBytes + 256));
    auto fail = [&](int code) {
        free_windows(D);
        return code;
    };
    auto body = [&]() -> int {
        MXW_TRY(mx::dev_malloc((void **)&D.window, (size_t)nWG * 8));
        MXW_TRY(hipMemsetAsync(counts.p, 0, 256 + 3 * countB, s));
        hipLaunchKernelGGL(window_rows_kernel, dim3((unsigned)std::min<long long>(kRowsBlocks, ((long long)rows + kBlock - 1) / kBlock)), dim3(kBlock), 0, s,
                           rowPtr_dev, rows, tot);
        MXW_TRY(hipGetLastError());
        hipLaunchKernelGGL(window_find_kernel, dim3(nWG), dim3(kBlock), 0, s, rowPtr_dev, col_dev, rows, cols, nChunks, waves, epv, widest,
                           (int2 *)D.window, units, farSteps, alone, tot);
        MXW_TRY(hipGetLastError());
        // (for the estimate below, before anything is waited for; from 8192 windows instead of a thousand: 30 us)
        long long sampled = 0;
        MXW_TRY(launch_lines_per_gather(dtype, nnz, col_dev, 1024, (unsigned long long *)(tot + 8), &sampled, s));
        int dev = 0, nCU = 0;
        MXW_TRY(hipGetDevice(&dev));
        MXW_TRY(hipDeviceGetAttribute(&nCU, hipDeviceAttributeMultiprocessorCount, dev));
        int h[10] = {0, 0, 0, 0, 0, 0, 0, 0, 0, 0};
        MXW_TRY(hipMemcpyAsync(h, tot, sizeof(h), hipMemcpyDeviceToHost, s));
        MXW_TRY(hipStreamSynchronize(s));
        const double stored = (double)h[1] * window_unit_bytes(f64) + (double)h[2] * 64 * (4 + es);
        if (h[0] || h[1] <= 0 || h[4] > kWindowFarMost * (double)nnz) return fail(MX_OK);
        unsigned long long lineSum = 0;
        std::memcpy(&lineSum, h + 8, 8);
        const double lines = sampled > 0 ? (double)lineSum / (double)sampled : 1.0;
        if (!window_form_pays(f64, nnz, stored, stored + ((double)rows + cols) * es, nWG, nCU, other_forms_us(dtype, rows, cols, nnz, lines)))
            return fail(MX_OK);
        if (f64 && nnz >= 65536 && mx::opt().csr_dict != 0) {
            // few distinct binary64 values: slices with a byte a value move a third of what this form would
            void *codes = nullptr;
            std::vector<unsigned char> dict;
            int nDict = 0;
            const int rc = value_dict_device(dtype, val_dev, nnz, 255, &codes, dict, &nDict, s);
            (void)mx::dev_free(codes);
            if (rc) return rc;
            if (nDict > 0) return fail(MX_OK);
        }
        D.rows = rows;
        D.cols = cols;
        D.nnz = nnz;
        D.nChunks = nChunks;
        D.nWG = nWG;
        D.units = h[1];
        D.farSteps = h[2];
        D.nApart = h[5];
        D.unitBytes = window_unit_bytes(f64);
        D.zeroPlace = h[3] * epv;
        D.ldsBytes = std::max((D.zeroPlace + epv) * es, 64 * kWindowWaves * 8);
        MXW_TRY(mx::dev_malloc((void **)&D.chunk, (size_t)nChunks * 16));
        MXW_TRY(mx::dev_malloc((void **)&D.stream, ((size_t)D.units + 1) * D.unitBytes));
        MXW_TRY(mx::dev_malloc((void **)&D.farCol, ((size_t)D.farSteps + 1) * 64 * 4));
        MXW_TRY(mx::dev_malloc(&D.farVal, ((size_t)D.farSteps + 1) * 64 * es));
        MXW_TRY(mx::dev_malloc((void **)&D.apart, ((size_t)D.nApart + 1) * 4));
        MXW_TRY(hipMemsetAsync(D.farCol + (size_t)D.farSteps * 64, 0xff, 64 * 4, s));  // the spare step: no entries
        MXW_TRY(rocprim::exclusive_scan(tmp.p, scanBytes, (const int *)units, (int *)unit0.p, 0, (size_t)nChunks + 1, rocprim::plus<int>(), s));
        MXW_TRY(rocprim::exclusive_scan(tmp.p, scanBytes, (const int *)farSteps, (int *)far0.p, 0, (size_t)nChunks + 1, rocprim::plus<int>(), s));
        MXW_TRY(rocprim::exclusive_scan(tmp.p, scanBytes, (const int *)alone, (int *)apart0.p, 0, (size_t)nChunks + 1, rocprim::plus<int>(), s));
        const dim3 grid((unsigned)((nChunks + kBlock / 64 - 1) / (kBlock / 64)));
        const int *U0 = (const int *)unit0.p, *F0 = (const int *)far0.p, *A0 = (const int *)apart0.p;
        if (f64)
            hipLaunchKernelGGL(window_fill_kernel<double>, grid, dim3(kBlock), 0, s, rowPtr_dev, col_dev, (const double *)val_dev,
                               (const int2 *)D.window, U0, F0, A0, rows, nChunks, waves, D.zeroPlace, (int4 *)D.chunk, D.stream, D.farCol,
                               (double *)D.farVal, D.apart);
        else
            hipLaunchKernelGGL(window_fill_kernel<_Float16>, grid, dim3(kBlock), 0, s, rowPtr_dev, col_dev, (const _Float16 *)val_dev,
                               (const int2 *)D.window, U0, F0, A0, rows, nChunks, waves, D.zeroPlace, (int4 *)D.chunk, D.stream, D.farCol,
                               (_Float16 *)D.farVal, D.apart);
        MXW_TRY(hipGetLastError());
        if (D.ldsBytes > 65536) {
            const void *fn[2] = {f64 ? window_kernel<double, false, kWindowWaves>() : window_kernel<_Float16, false, kWindowWaves>(),
                                 f64 ? window_kernel<double, true, kWindowWaves>() : window_kernel<_Float16, true, kWindowWaves>()};
            for (const void *f : fn) MXW_TRY(hipFuncSetAttribute(f, hipFuncAttributeMaxDynamicSharedMemorySize, kWindowBytesMost + 1024));
        }
        MXW_TRY(hipStreamSynchronize(s));
        return MX_OK;
    };
    const int rc = body();
    return rc ? fail(rc) : rc;
}

hipError_t launch_windows(mx_dtype dtype, const DeviceWindows &D, const void *x, void *y, hipStream_t s)
{
    if (D.nChunks <= 0) return hipSuccess;
#define MX_LAUNCH_WINDOWS(VT, KEEP)                                                                                                          \
    hipLaunchKernelGGL((mxw::csr_window_kernel<VT, KEEP, kWindowWaves>), dim3(D.nWG + D.nApart), dim3(64 * kWindowWaves), D.ldsBytes, s,                  \
                       (const int2 *)D.window, (const int4 *)D.chunk, (const unsigned char *)D.stream, (const int *)D.farCol,                  \
                       (const VT *)D.farVal, (const int *)D.apart, (const VT *)x, (VT *)y, D.rows, D.cols, D.nChunks, D.nApart,               \
                       D.zeroPlace)
    if (dtype == MX_F64) {
        if (D.keep) MX_LAUNCH_WINDOWS(double, true);
        else MX_LAUNCH_WINDOWS(double, false);
    } else {
        if (D.keep) MX_LAUNCH_WINDOWS(_Float16, true);
        else MX_LAUNCH_WINDOWS(_Float16, false);
    }
#undef MX_LAUNCH_WINDOWS
    return hipGetLastError();
}

}  // namespace mx

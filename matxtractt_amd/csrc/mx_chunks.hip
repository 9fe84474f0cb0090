// Which workgroup and which wave streams which chunk of a slice layout, decided on the device: the same decisions, and the
// same arrays, as plan_slice_chunks (mx_host_layout.cpp) makes on the host.
//
// What there is to do is small -- a chunk is 64 virtual rows -- but serial by nature: every chunk goes to the
// workgroup with the least work so far, longest first, and inside the workgroup to such a wave.  Made on the host
// it cost two waits, the lengths' way down, seven arrays' way up and the dealing itself, during all of which the device had nothing
// to do: 0.8 of the 2.2 ms that the plan of 7.6 million binary64 entries (17 thousand chunks) took, 1.7 of 3.1 with 57 thousand chunks; so it is 0.15.  The serial part is cut down
// in two ways.  Chunks of one length are dealt together: how many of them each workgroup gets follows from the level that
// its load is filled up to, which is searched for (a wave, its lanes holding the workgroups' loads); and slices, then
// workgroups, are dealt independently of each other, a wave each.
#include "mx_chunks.h"

#include <algorithm>

#include <rocprim/device/device_scan.hpp>

#include "mx_digits.h"

namespace mxl {

constexpr int W = mx::kSliceWaves;
constexpr int kCost = mx::kSliceChunkCost;
constexpr int kCapMost = 4096;     // entries of a virtual row at most (the layout's cap)
constexpr int kBinsLds = 1024;     // workgroups of a slice whose loads are kept in LDS; more of them in memory
constexpr int kFewChunks = 8;      // so many chunks of one length go one by one

// DPP moves: lane i takes lane i - n of its row of sixteen (or the last of the rows before); lanes without a source keep `old`.
template <int CTRL, int ROWS>
__device__ __forceinline__ int dpp_from(int old, int v)
{
    return __builtin_amdgcn_update_dpp(old, v, CTRL, ROWS, 0xf, false);
}
template <typename F>
__device__ __forceinline__ int wave_reduce(int v, F f)  // the result of all lanes, in every lane
{
    v = f(v, dpp_from<0x111, 0xf>(v, v));  // row_shr 1, 2, 4, 8: idempotent or masked by the caller's neutral element
    v = f(v, dpp_from<0x112, 0xf>(v, v));
    v = f(v, dpp_from<0x114, 0xf>(v, v));
    v = f(v, dpp_from<0x118, 0xf>(v, v));
    v = f(v, dpp_from<0x142, 0xa>(v, v));  // row_bcast 15, 31
    v = f(v, dpp_from<0x143, 0xc>(v, v));
    return __builtin_amdgcn_readlane(v, 63);
}
__device__ __forceinline__ int wave_min(int v)
{
    return wave_reduce(v, [](int a, int b) { return min(a, b); });
}
__device__ __forceinline__ int wave_max(int v)
{
    return wave_reduce(v, [](int a, int b) { return max(a, b); });
}
// running sums: lane i gets the sum of lanes 0 .. i
__device__ __forceinline__ int wave_scan(int v)
{
    v += dpp_from<0x111, 0xf>(0, v);
    v += dpp_from<0x112, 0xf>(0, v);
    v += dpp_from<0x114, 0xf>(0, v);
    v += dpp_from<0x118, 0xf>(0, v);
    v += dpp_from<0x142, 0xa>(0, v);
    v += dpp_from<0x143, 0xc>(0, v);
    return v;
}

struct Totals {
    long long steps, chunks;
    int nWG, maxWgChunks;
    int refused, crowded, most, maxWgGroups;  // (one-launch form; a launch that raises one of the first two does not read it)
};

// sliceStart[q] = virtual rows of the slices before q, chunkBase[q] = chunks of those, for q in [0, S]; work[q] cleared.
__global__ __launch_bounds__(1024) void slice_chunks_kernel(const unsigned *__restrict__ sortedKey, int nV, int S, unsigned perSlice,
                                                            int *__restrict__ sliceStart, int *__restrict__ chunkBase,
                                                            unsigned long long *__restrict__ work)
{
    __shared__ int part[16];
    const int tid = threadIdx.x, per = (S + 1023) / 1024, q0 = min(S, tid * per), q1 = min(S, q0 + per);
    auto first = [&](int q) {  // position whose key is not below the slice's first
        const unsigned long long want = (unsigned long long)q * perSlice;
        int lo = 0, hi = nV;
        while (lo < hi) {
            const int mid = lo + (hi - lo) / 2;
            if ((unsigned long long)sortedKey[mid] < want) lo = mid + 1;
            else hi = mid;
        }
        return lo;
    };
    int n = 0, a = first(q0);
    for (int q = q0; q < q1; ++q) {
        const int z = first(q + 1);
        sliceStart[q] = a;
        n += (z - a + 63) / 64;
        a = z;
    }
    if (q1 == S) sliceStart[S] = nV;  // (every key belongs to a slice)
    const int run = wave_scan(n);
    if ((tid & 63) == 63) part[tid >> 6] = run;
    __syncthreads();
    int at = run - n;
    for (int w = 0; w < (tid >> 6); ++w) at += part[w];
    for (int q = q0; q < q1; ++q) {
        chunkBase[q] = at;
        work[q] = 0;
        at += ((q + 1 < q1 ? sliceStart[q + 1] : a) - sliceStart[q] + 63) / 64;
        if (q == S - 1) chunkBase[S] = at;
    }
}

// Of every chunk its first virtual row, their number and its steps; work[q] += what the chunks of slice q cost.
__global__ __launch_bounds__(kBlock) void chunk_steps_kernel(const int *__restrict__ sliceStart, const int *__restrict__ chunkBase, int S,
                                                             const int *__restrict__ sorted, const int *__restrict__ vLen, int *__restrict__ first,
                                                             int *__restrict__ number, int *__restrict__ steps, unsigned long long *__restrict__ work)
{
    const int c = blockIdx.x * kBlock + threadIdx.x, lane = threadIdx.x & 63;
    const bool in = c < chunkBase[S];
    int q = -1, len = 0;
    if (in) {
        int lo = 0, hi = S - 1;  // the last slice whose chunks begin at or before c
        while (lo < hi) {
            const int mid = (lo + hi + 1) >> 1;
            if (chunkBase[mid] <= c) lo = mid;
            else hi = mid - 1;
        }
        q = lo;
        const int f = sliceStart[q] + 64 * (c - chunkBase[q]);
        len = vLen[sorted[f]];
        first[c] = f;
        number[c] = min(64, sliceStart[q + 1] - f);
        steps[c] = len;
    }
    const int one = __builtin_amdgcn_readfirstlane(q);
    if (__all(q == one)) {  // (nearly always: one atomic for the wave)
        const int sum = __builtin_amdgcn_readlane(wave_scan(in ? len + kCost : 0), 63);
        if (lane == 0 && one >= 0) atomicAdd(&work[one], (unsigned long long)sum);
    } else if (in) {
        atomicAdd(&work[q], (unsigned long long)(len + kCost));
    }
}

// The workgroups of every slice, in proportion to its work (largest remainders, at least one where there is anything): wgBase.
__global__ __launch_bounds__(64) void slice_shares_kernel(const unsigned long long *__restrict__ work, const int *__restrict__ chunkBase, int S,
                                                          int budget, double *__restrict__ missing, int *__restrict__ groups, int *__restrict__ wgBase,
                                                          Totals *__restrict__ totals)
{
    // (missing: share less workgroups; a lane has its own slices' part of both arrays)
    const int lane = threadIdx.x, per = (S + 63) / 64, q0 = min(S, lane * per), q1 = min(S, q0 + per);
    unsigned long long all = 0;
    int busy = 0;
    for (int q = q0; q < q1; ++q) {
        all += work[q];
        busy += chunkBase[q + 1] > chunkBase[q];
    }
    for (int off = 32; off; off >>= 1) {
        all += __shfl_xor(all, off);
        busy += __shfl_xor(busy, off);
    }
    const int total = max(budget, busy);
    int used = 0;
    for (int q = q0; q < q1; ++q) {
        const bool some = chunkBase[q + 1] > chunkBase[q];
        const double want = some ? (double)(long long)work[q] * total / (double)(long long)all : 0.0;
        groups[q] = some ? max(1, (int)want) : 0;
        missing[q] = some ? want - groups[q] : -1e300;
        used += groups[q];
    }
    for (int off = 32; off; off >>= 1) used += __shfl_xor(used, off);
    for (; used < total && busy > 0; ++used) {  // what rounding down left over goes where most is missing
        double most = -1e301;
        int best = S;
        for (int q = q0; q < q1; ++q)
            if (missing[q] > most) {
                most = missing[q];
                best = q;
            }
        for (int off = 32; off; off >>= 1) {
            const double m = __shfl_xor(most, off);
            const int b = __shfl_xor(best, off);
            if (m > most || (m == most && b < best)) {
                most = m;
                best = b;
            }
        }
        if (best >= q0 && best < q1) {
            // (as the host: the share itself less the workgroups it has now)
            const double want = (double)(long long)work[best] * total / (double)(long long)all;
            ++groups[best];
            missing[best] = want - groups[best];
        }
    }
    int mine = 0;
    for (int q = q0; q < q1; ++q) {
        const int nc = chunkBase[q + 1] - chunkBase[q];
        groups[q] = nc ? min(max(groups[q], (nc + mx::kSliceWgChunks - 1) / mx::kSliceWgChunks), nc) : 0;
        mine += groups[q];
    }
    int at = wave_scan(mine) - mine;
    for (int q = q0; q < q1; ++q) {
        wgBase[q] = at;
        at += groups[q];
    }
    if (lane == 63) {
        wgBase[S] = at;
        totals->nWG = at;
        totals->chunks = chunkBase[S];
    }
}

// The chunks of slice blockIdx.x to its workgroups: those of one length together, each to the workgroup with the least work so far (the
// first of equals), a workgroup's share of them consecutive.  list[wgChunk[b] ..] are the chunks of workgroup b in the order they
// are dealt, wgSlice[b] its slice.
__global__ __launch_bounds__(64) void deal_slices_kernel(const int *__restrict__ steps, const int *__restrict__ chunkBase, const int *__restrict__ wgBase,
                                                         int *__restrict__ binMem, int *__restrict__ whose, int *__restrict__ place,
                                                         int *__restrict__ wgSlice, int *__restrict__ wgChunk, int *__restrict__ list)
{
    __shared__ int ofLength[kCapMost + 1];
    __shared__ int binLds[3 * kBinsLds];
    const int q = blockIdx.x, lane = threadIdx.x, c0 = chunkBase[q], c1 = chunkBase[q + 1], b0 = wgBase[q], G = wgBase[q + 1] - b0;
    if (G == 0) return;
    for (int i = lane; i <= kCapMost; i += 64) ofLength[i] = 0;
    // (lane l holds the workgroups [l * per, (l + 1) * per), so that the first lane of equals has the first of them)
    const int per = (G + 63) / 64, g0 = min(G, lane * per), g1 = min(G, g0 + per);
    int *load = G <= kBinsLds ? binLds : binMem + 3 * (size_t)b0, *had = load + G, *take = had + G;
    for (int g = g0; g < g1; ++g) load[g] = had[g] = 0;
    __syncthreads();
    for (int c = c0 + lane; c < c1; c += 64) atomicAdd(&ofLength[min(steps[c], kCapMost)], 1);
    __syncthreads();
    int at = c0;
    for (int len = kCapMost; len >= 0; --len) {
        // the next length that there is, 64 at a look
        {
            const unsigned long long m = __ballot(len - lane >= 0 && ofLength[max(len - lane, 0)] > 0);
            if (!m) {
                len -= 63;
                continue;
            }
            len -= __builtin_ctzll(m);
        }
        const int n = ofLength[len], w = len + kCost;
        for (int g = g0; g < g1; ++g) take[g] = 0;
        if (n <= kFewChunks) {
            for (int k = 0; k < n; ++k) {
                int least = 0x7fffffff, best = -1;
                for (int g = g0; g < g1; ++g)
                    if (had[g] + take[g] < mx::kSliceWgChunks && load[g] < least) {
                        least = load[g];
                        best = g;
                    }
                const unsigned long long m = __ballot(least == wave_min(least));
                if (lane == __builtin_ctzll(m) && best >= 0) {
                    ++take[best];
                    load[best] += w;
                }
            }
        } else {
            // The level: the highest T for which at most n chunks begin below it when every workgroup is filled up, chunk by chunk,
            // from its load; those that begin at T exactly go to the first workgroups.
            const double inverse = 1.0 / w;
            auto below = [&](int g, int T) {  // chunks of workgroup g that begin below T
                const int d = T - load[g];
                return d <= 0 ? 0 : min((int)((d + w - 1 + 0.5) * inverse), mx::kSliceWgChunks - had[g]);
            };
            int lo = 0x7fffffff, top = 0, fullest = 0, sum = 0;
            for (int g = g0; g < g1; ++g) {
                lo = min(lo, load[g]);
                top = max(top, load[g]);
                fullest = max(fullest, had[g]);
                sum += load[g];
            }
            lo = wave_min(lo);
            top = wave_max(top);
            fullest = wave_max(fullest);
            // (no workgroup is full before the others: the level lies within a chunk of the mean)
            long long total = sum;
            for (int off = 32; off; off >>= 1) total += __shfl_xor(total, off);
            long long hi = (total + (long long)n * w) / G + w + 1;
            if (fullest + (hi - lo) / w + 2 >= mx::kSliceWgChunks) hi = top + (long long)mx::kSliceWgChunks * w + 1;  // (all are full)
            long long a = max((long long)lo, (total + (long long)n * w) / G - (top - lo) - w), z = hi;  // below(a) <= n, below(z + 1) > n or z = hi
            auto count = [&](long long T) {
                int k = 0;
                for (int g = g0; g < g1; ++g) k += below(g, (int)T);
                return __builtin_amdgcn_readlane(wave_scan(k), 63);
            };
            if (count(a) > n) a = lo;
            while (a < z) {
                const long long mid = a + (z - a + 1) / 2;
                if (count(mid) <= n) a = mid;
                else z = mid - 1;
            }
            const int T = (int)a;
            int mine = 0, more = 0;
            for (int g = g0; g < g1; ++g) {
                const int k = below(g, T);
                take[g] = k;
                mine += k;
                more += load[g] + k * w == T && had[g] + k < mx::kSliceWgChunks;
            }
            const int rest = n - __builtin_amdgcn_readlane(wave_scan(mine), 63);
            int seen = wave_scan(more) - more;
            for (int g = g0; g < g1; ++g) {
                const bool next = load[g] + take[g] * w == T && had[g] + take[g] < mx::kSliceWgChunks;
                if (next && seen++ < rest) ++take[g];
                load[g] += take[g] * w;
            }
        }
        int mine = 0;
        for (int g = g0; g < g1; ++g) mine += take[g];
        int c = at + wave_scan(mine) - mine;
        for (int g = g0; g < g1; ++g) {
            for (int k = 0; k < take[g]; ++k, ++c) {
                whose[c] = g;
                place[c] = had[g] + k;
            }
            had[g] += take[g];
        }
        at += n;
    }
    int mine = 0;
    for (int g = g0; g < g1; ++g) mine += had[g];
    int first = c0 + wave_scan(mine) - mine;
    for (int g = g0; g < g1; ++g) {
        const int n = had[g];
        wgSlice[b0 + g] = q;
        wgChunk[b0 + g] = had[g] = first;
        first += n;
    }
    __syncthreads();
    for (int c = c0 + lane; c < c1; c += 64) list[had[whose[c]] + place[c]] = c;
}

// The chunks of workgroup blockIdx.x to its waves: each to the wave with the least work so far.  Chunks get their final numbers; steps are
// counted from the workgroup's first.
__global__ __launch_bounds__(64) void deal_waves_kernel(const Totals *__restrict__ totals, const int *__restrict__ wgChunk, const int *__restrict__ list,
                                                        const int *__restrict__ first, const int *__restrict__ number, const int *__restrict__ steps,
                                                        int SPB, int *__restrict__ how, int *__restrict__ chunkFirst, int *__restrict__ chunkN,
                                                        int *__restrict__ chunkSteps, int *__restrict__ chunkEnd, int *__restrict__ chunkAt,
                                                        int *__restrict__ wave4, int *__restrict__ wgSteps, int *__restrict__ wgChunks)
{
    const int b = blockIdx.x, lane = threadIdx.x;
    if (b >= totals->nWG) return;
    const int c0 = wgChunk[b], n = (b + 1 < totals->nWG ? wgChunk[b + 1] : (int)totals->chunks) - c0;
    // (lanes 0 .. W - 1 are the waves)
    int cost = lane < W ? 0 : 0x7fffffff, run = 0, had = 0;
    for (int k0 = 0; k0 < n; k0 += 64) {
        const int len = k0 + lane < n ? steps[list[c0 + k0 + lane]] : 0, m = min(64, n - k0);
        int w_ = 0, at_ = 0, num_ = 0;
        for (int k = 0; k < m; ++k) {
            const int l = __builtin_amdgcn_readlane(len, k);
            int least = min(cost, dpp_from<0x111, 0xf>(0x7fffffff, cost));
            least = min(least, dpp_from<0x112, 0xf>(0x7fffffff, least));
            least = min(least, dpp_from<0x114, 0xf>(0x7fffffff, least));
            least = __builtin_amdgcn_readlane(least, W - 1);
            const int best = __builtin_ctzll(__ballot(cost == least));
            const int at = __builtin_amdgcn_readlane(run, best), num = __builtin_amdgcn_readlane(had, best);
            if (lane == k) {
                w_ = best;
                at_ = at;
                num_ = num;
            }
            if (lane == best) {
                cost += l + kCost;
                run += l;
                ++had;
            }
        }
        if (k0 + lane < n) {
            how[3 * (size_t)(c0 + k0 + lane)] = w_;
            how[3 * (size_t)(c0 + k0 + lane) + 1] = at_;
            how[3 * (size_t)(c0 + k0 + lane) + 2] = num_;
        }
    }
    const int stored = lane < W ? (run + SPB - 1) / SPB * SPB : 0, chunks = lane < W ? had : 0;
    const int stepAt = wave_scan(stored) - stored, chunkBefore = wave_scan(chunks) - chunks;
    if (lane < W) {
        int *d = wave4 + ((size_t)b * W + lane) * 4;
        d[0] = stepAt;
        d[1] = stored / SPB;
        d[2] = chunkBefore;
        d[3] = chunks;
    }
    if (lane == W - 1) {
        wgSteps[b] = stepAt + stored;
        wgChunks[b] = n;
    }
    __syncthreads();
    for (int k0 = 0; k0 < n; k0 += 64) {
        const bool in = k0 + lane < n;
        const int k = min(k0 + lane, n - 1);
        const int w = how[3 * (size_t)(c0 + k)], at = how[3 * (size_t)(c0 + k) + 1], num = how[3 * (size_t)(c0 + k) + 2], c = list[c0 + k];
        const int to = c0 + __shfl(chunkBefore, w) + num, a = __shfl(stepAt, w) + at, len = steps[c];
        if (!in) continue;
        chunkFirst[to] = first[c];
        chunkN[to] = number[c];
        chunkSteps[to] = len;
        chunkEnd[to] = at + len;
        chunkAt[to] = a;
    }
}

// wgStep[b] = steps of the workgroups before b; the totals.
__global__ __launch_bounds__(1024) void wg_steps_kernel(const int *__restrict__ wgSteps, const int *__restrict__ wgChunks, long long *__restrict__ wgStep,
                                                        Totals *__restrict__ totals)
{
    __shared__ long long part[16];
    __shared__ int most[16];
    const int tid = threadIdx.x, lane = tid & 63, n = totals->nWG;
    long long before = 0;
    int top = 0;
    for (int b0 = 0; b0 < n; b0 += 1024) {
        const int b = b0 + tid;
        const long long v = b < n ? wgSteps[b] : 0;
        long long run = v;
        for (int off = 1; off < 64; off <<= 1) {
            const long long o = __shfl_up(run, off);
            if (lane >= off) run += o;
        }
        if (lane == 63) part[tid >> 6] = run;
        __syncthreads();
        long long pre = before;
        for (int w = 0; w < 16; ++w) {
            if (w < (tid >> 6)) pre += part[w];
            before += part[w];
        }
        if (b < n) {
            wgStep[b] = pre + run - v;
            top = max(top, wgChunks[b]);
        }
        __syncthreads();
    }
    top = wave_max(top);
    if (lane == 0) most[tid >> 6] = top;
    __syncthreads();
    if (tid == 0) {
        for (int w = 1; w < 16; ++w) top = max(top, most[w]);
        totals->steps = before;
        totals->maxWgChunks = top;
    }
}

// The descriptors, and the chunks' first steps in the streams.
__global__ __launch_bounds__(64) void emit_chunks_kernel(int nWG, int SPB, const int *__restrict__ wgSlice, const int *__restrict__ wgChunk,
                                                         const int *__restrict__ wgChunks, const long long *__restrict__ wgStep,
                                                         const int *__restrict__ wave4, const int *__restrict__ chunkEndIn,
                                                         const int *__restrict__ chunkAt, int totalChunks, int *__restrict__ wgDesc,
                                                         int *__restrict__ waveDesc, int *__restrict__ chunkEnd, long long *__restrict__ chunkStep0)
{
    const int b = blockIdx.x, lane = threadIdx.x;
    if (b >= nWG) {  // the padding
        if (lane < 4) wgDesc[(size_t)nWG * 4 + lane] = waveDesc[(size_t)nWG * W * 4 + lane] = 0;
        chunkEnd[totalChunks + lane] = 0;
        return;
    }
    const int c0 = wgChunk[b], n = wgChunks[b];
    const long long step0 = wgStep[b];
    if (lane < 4) wgDesc[(size_t)b * 4 + lane] = lane == 0 ? wgSlice[b] : lane == 1 ? c0 : lane == 2 ? n : 0;
    if (lane < W * 4) {
        const int v = wave4[(size_t)b * W * 4 + lane];
        waveDesc[(size_t)b * W * 4 + lane] = lane % 4 == 0 ? (int)((step0 + v) / SPB) : v;
    }
    for (int c = c0 + lane; c < c0 + n; c += 64) {
        chunkEnd[c] = chunkEndIn[c];
        chunkStep0[c] = step0 + chunkAt[c];
    }
}
static_assert(W * 4 <= 64 && W <= 8, "a wave writes a workgroup's descriptors, eight lanes are its waves");

// The arrays of a plan on its way: at most N chunks and G workgroups.
struct Dealing {
    Buf scratch;
    int *first, *number, *steps, *list, *how, *chunkEnd;              // chunks in the order they are dealt
    int *wgSlice, *wgChunk, *wgSteps, *wgChunks, *wave4;              // workgroups
    int *chunkFirst, *chunkN, *chunkSteps, *chunkAt;                  // chunks in their final numbering (in P.made)
    long long *wgStep, *chunkStep0;
    Totals *totals;
    Totals got{};
    size_t N = 0, G = 0;

    static size_t al(size_t b) { return (b + 255) & ~(size_t)255; }
    unsigned char *at = nullptr;
    template <typename T>
    T *part(size_t n)
    {
        T *q = (T *)at;
        at += al(n * sizeof(T));
        return q;
    }
    // `more` bytes behind, for the caller's own (part)
    int make(size_t n, size_t g, size_t more, ChunkPlan &P)
    {
        N = n + 1;
        G = g + 1;
        MXL_TRY(mx::dev_malloc(&scratch.p, 7 * al(N * 4) + al(3 * N * 4) + 4 * al(G * 4) + al(G * W * 16) + al(G * 8) + al(sizeof(Totals)) + more));
        MXL_TRY(mx::dev_malloc(&P.made.p, 4 * al(N * 4) + al(N * 8)));
        at = (unsigned char *)P.made.p;
        chunkFirst = part<int>(N), chunkN = part<int>(N), chunkSteps = part<int>(N), chunkAt = part<int>(N), chunkStep0 = part<long long>(N);
        at = (unsigned char *)scratch.p;
        first = part<int>(N), number = part<int>(N), steps = part<int>(N), list = part<int>(N), chunkEnd = part<int>(N), how = part<int>(3 * N);
        wgSlice = part<int>(G), wgChunk = part<int>(G), wgSteps = part<int>(G), wgChunks = part<int>(G), wave4 = part<int>(G * W * 4);
        wgStep = part<long long>(G);
        totals = part<Totals>(1);
        return MX_OK;
    }
    // The chunks of every workgroup to its waves, and the totals to the host.
    int deal(int SPB, hipStream_t s)
    {
        hipLaunchKernelGGL(deal_waves_kernel, dim3((unsigned)G), dim3(64), 0, s, (const Totals *)totals, (const int *)wgChunk, (const int *)list, (const int *)first,
                           (const int *)number, (const int *)steps, SPB, how, chunkFirst, chunkN, chunkSteps, chunkEnd, chunkAt, wave4, wgSteps, wgChunks);
        hipLaunchKernelGGL(wg_steps_kernel, dim3(1), dim3(1024), 0, s, (const int *)wgSteps, (const int *)wgChunks, wgStep, totals);
        MXL_TRY(hipGetLastError());
        MXL_TRY(hipMemcpyAsync(&got, totals, sizeof(got), hipMemcpyDeviceToHost, s));
        MXL_TRY(hipStreamSynchronize(s));
        return MX_OK;
    }
    int emit(int SPB, ChunkPlan &P, hipStream_t s)
    {
        if (got.steps * 64 > 2000000000LL || got.chunks * 64 > 2000000000LL) {
            mx::set_error("slice layout: too many entries for 32-bit offsets");
            return MX_ERR_ARG;
        }
        P.nWG = got.nWG;
        P.maxWgChunks = got.maxWgChunks;
        P.totalSteps = got.steps;
        P.totalChunks = got.chunks;
        MXL_TRY(mx::dev_malloc(&P.wgDesc.p, ((size_t)P.nWG * 4 + 4) * 4));
        MXL_TRY(mx::dev_malloc(&P.waveDesc.p, ((size_t)P.nWG * W * 4 + 4) * 4));
        MXL_TRY(mx::dev_malloc(&P.chunkEnd.p, ((size_t)P.totalChunks + 64) * 4));
        hipLaunchKernelGGL(emit_chunks_kernel, dim3((unsigned)P.nWG + 1), dim3(64), 0, s, P.nWG, SPB, (const int *)wgSlice, (const int *)wgChunk,
                           (const int *)wgChunks, (const long long *)wgStep, (const int *)wave4, (const int *)chunkEnd, (const int *)chunkAt, (int)P.totalChunks,
                           P.wgDesc.as<int>(), P.waveDesc.as<int>(), P.chunkEnd.as<int>(), chunkStep0);
        MXL_TRY(hipGetLastError());
        P.chunkFirst = chunkFirst;
        P.chunkN = chunkN;
        P.chunkSteps = chunkSteps;
        P.chunkStep0 = chunkStep0;
        return MX_OK;  // (the scratch goes back to the scope, whose next request is served in the order of the stream)
    }
};

int plan_chunks_device(mx_dtype dtype, int budget, int S, int nV, const unsigned *sortedKey, unsigned perSlice, const int *sorted,
                       const int *vLen, ChunkPlan &P, hipStream_t s)
{
    const int SPB = mx::kSliceBatchEntries / mx::slice_step_entries(dtype);
    const long long chunksMost = (long long)nV / 64 + S;
    const size_t N = (size_t)chunksMost, G = (size_t)budget + 2 * (size_t)S + (size_t)(chunksMost / mx::kSliceWgChunks) + 1, n1 = (size_t)S + 1;
    Dealing D;
    int rc = D.make(N, G, 4 * D.al(n1 * 4) + 2 * D.al(n1 * 8) + 2 * D.al(N * 4) + D.al(3 * G * 4), P);
    if (rc) return rc;
    int *sliceStart = D.part<int>(n1), *chunkBase = D.part<int>(n1), *wgBase = D.part<int>(n1), *groups = D.part<int>(n1);
    unsigned long long *work = D.part<unsigned long long>(n1);
    double *missing = D.part<double>(n1);
    int *whose = D.part<int>(N), *place = D.part<int>(N), *bins = D.part<int>(3 * G);
    hipLaunchKernelGGL(slice_chunks_kernel, dim3(1), dim3(1024), 0, s, sortedKey, nV, S, perSlice, sliceStart, chunkBase, work);
    hipLaunchKernelGGL(chunk_steps_kernel, grid(chunksMost), dim3(kBlock), 0, s, (const int *)sliceStart, (const int *)chunkBase, S, sorted, vLen, D.first, D.number,
                       D.steps, work);
    hipLaunchKernelGGL(slice_shares_kernel, dim3(1), dim3(64), 0, s, (const unsigned long long *)work, (const int *)chunkBase, S, budget, missing, groups,
                       wgBase, D.totals);
    hipLaunchKernelGGL(deal_slices_kernel, dim3((unsigned)S), dim3(64), 0, s, (const int *)D.steps, (const int *)chunkBase, (const int *)wgBase, bins, whose, place,
                       D.wgSlice, D.wgChunk, D.list);
    MXL_TRY(hipGetLastError());
    if ((rc = D.deal(SPB, s))) return rc;
    return D.emit(SPB, P, s);
}

// ---- the one-launch form ----
// The decisions of plan_fused (mx_host_layout.cpp), on the device: the same arrays.  Virtual rows are put in order by (XCD, slice), which
// with the running sum of their lengths gives every one its workgroup; a workgroup's virtual rows, in a row of that order, are
// put in order by length in LDS.  (250 thousand virtual rows: on the host, with the records' way down and the
// plan's way up, 3.9 ms; so 0.2.)
constexpr int X = mx::kFusedXcds, GR = mx::kFusedGroupRows, kWgChunks = mx::kFusedWgChunks;
static_assert(kWgChunks * 64 <= mxd::kTile, "a workgroup's virtual rows are put in order at once");
struct Parts {
    int S, rows, nGroups, nk, nV, cap;
    const int *vRow, *vSlice, *vLen;
    int *xg;  // [X + 1] first group of every XCD
    __device__ __forceinline__ int of(int t) const
    {
        const int g = vRow[t] / GR;
        int k = 0;
#pragma unroll
        for (int i = 1; i < X; ++i) k += xg[i] <= g;
        return k * S + vSlice[t];
    }
};

__global__ __launch_bounds__(kBlock) void most_vrows_kernel(const int *__restrict__ segPtr, int rows, Totals *__restrict__ totals)
{
    int m = 0;
    for (long long r = (long long)blockIdx.x * kBlock + threadIdx.x; r < rows; r += (long long)gridDim.x * kBlock) m = max(m, segPtr[r + 1] - segPtr[r]);
    m = wave_max(m);
    if ((threadIdx.x & 63) == 0 && m > *(volatile int *)&totals->most) atomicMax(&totals->most, m);
}

// The groups of every XCD: an eighth of the entries each, one group at least.
__global__ __launch_bounds__(64) void xcd_groups_kernel(const int *__restrict__ rowPtr, long long nnz, Parts P, Totals *__restrict__ totals)
{
    const int lane = threadIdx.x;
    const long long target = nnz * lane / X;
    int lo = 0, hi = P.nGroups;
    while (lo < hi) {  // the first group that begins at or behind the target
        const int mid = (lo + hi) >> 1;
        if ((long long)rowPtr[min(P.rows, mid * GR)] < target) lo = mid + 1;
        else hi = mid;
    }
    int x = 0;
    if (lane == 0) P.xg[0] = 0;
    for (int k = 1; k < X; ++k) {
        const int g = max(x, __builtin_amdgcn_readlane(lo, k));
        x = min(max(g, x + 1), P.nGroups - (X - k));
        if (lane == 0) P.xg[k] = x;
    }
    if (lane == 0) {
        P.xg[X] = P.nGroups;
        totals->refused = totals->most > mx::kSliceLightSegs;  // (the form has so many places for a row's sums)
    }
}

// count[tile][part] virtual rows
__global__ __launch_bounds__(mxd::kThreads) void part_counts_kernel(Parts P, int tiles, int *__restrict__ count)
{
    __shared__ int here[mxd::kDigits];
    const int t = mxd::tile_of_block(tiles), tid = threadIdx.x, n = X * P.S;
    if (t >= tiles) return;
    for (int k = tid; k < n; k += mxd::kThreads) here[k] = 0;
    __syncthreads();
    for (int i = tid; i < mxd::kTile && t * mxd::kTile + i < P.nV; i += mxd::kThreads) {
        const int p = P.of(t * mxd::kTile + i), one = __builtin_amdgcn_readfirstlane(p);
        const unsigned long long same = __ballot(p == one);
        if ((tid & 63) == __builtin_ctzll(same)) atomicAdd(&here[one], __popcll(same));
        if (p != one) atomicAdd(&here[p], 1);
    }
    __syncthreads();
    for (int k = tid; k < n; k += mxd::kThreads) count[(size_t)t * n + k] = here[k];
}
// order[i]: the virtual rows by part, those of a part in the order of the rows; length[i] and part[i] of each
__global__ __launch_bounds__(mxd::kThreads, 8) void part_order_kernel(Parts P, int bits, int tiles, const int *__restrict__ before,
                                                                      const int *__restrict__ first, int *__restrict__ order, int *__restrict__ length,
                                                                      unsigned short *__restrict__ partOf)
{
    using namespace mxd;
    __shared__ Digits digits;
    __shared__ int start[kDigits];
    const int t = tile_of_block(tiles), tid = threadIdx.x, lane = tid & 63, w = tid >> 6, n = X * P.S;
    if (t >= tiles) return;
    const int t0 = t * kTile, size = min(kTile, P.nV - t0);
    for (int k = tid; k < n; k += kThreads) start[k] = first[k] + before[(size_t)t * n + k];
    int d[kPer], at[kPer];
#pragma unroll
    for (int j = 0; j < kPer; ++j) d[j] = P.of(t0 + min(w * kWave + j * 64 + lane, size - 1));
    place_by_digit<false>([&](int j) { return d[j]; }, size, bits, digits, start, (int *)nullptr, at);
#pragma unroll
    for (int j = 0; j < kPer; ++j) {
        const int i = w * kWave + j * 64 + lane;
        if (i >= size) continue;
        order[at[j]] = t0 + i;
        length[at[j]] = P.vLen[t0 + i];
        partOf[at[j]] = (unsigned short)d[j];
    }
}

// The workgroups of every part of XCD blockIdx.x, in proportion to its entries: partWgs, and the first of each: partBase.
__global__ __launch_bounds__(64) void part_shares_kernel(Parts P, const int *__restrict__ first, const int *__restrict__ run, double *__restrict__ want,
                                                         int *__restrict__ partWgs, int *__restrict__ partBase, Totals *__restrict__ totals)
{
    const int k = blockIdx.x, lane = threadIdx.x, per = (P.S + 63) / 64, q0 = min(P.S, lane * per), q1 = min(P.S, q0 + per), nk = P.nk;
    const int *f = first + (size_t)k * P.S;
    double *wanted = want + (size_t)k * P.S;
    int *wgs = partWgs + (size_t)k * P.S, *base = partBase + (size_t)k * P.S;
    const long long entries = (long long)run[f[P.S]] - run[f[0]];
    int busy = 0;
    for (int q = q0; q < q1; ++q) busy += f[q + 1] > f[q];
    busy = __builtin_amdgcn_readlane(wave_scan(busy), 63);
    if (busy == 0 || busy > nk) {
        if (lane == 0) atomicOr(&totals->refused, 1);
        return;
    }
    int used = 0;
    for (int q = q0; q < q1; ++q) {
        wgs[q] = 0;
        wanted[q] = 0.0;
        const int rows = f[q + 1] - f[q];
        if (rows == 0) continue;
        wanted[q] = (double)((long long)run[f[q + 1]] - run[f[q]]) * nk / (double)entries;
        wgs[q] = min(max(1, (int)wanted[q]), rows);
        used += wgs[q];
    }
    used = __builtin_amdgcn_readlane(wave_scan(used), 63);
    // the part whose `worth` is the highest (the first of equals) takes `step` workgroups; false: there is none
    auto change = [&](auto may, auto worth, int step) {
        double most = -1e300;
        int best = P.S;
        for (int q = q0; q < q1; ++q)
            if (may(q) && worth(q) > most) {
                most = worth(q);
                best = q;
            }
        for (int off = 32; off; off >>= 1) {
            const double m = __shfl_xor(most, off);
            const int b = __shfl_xor(best, off);
            if (m > most || (m == most && b < best)) {
                most = m;
                best = b;
            }
        }
        if (best >= q0 && best < q1) wgs[best] += step;
        return best < P.S;
    };
    for (; used > nk; --used)  // rounding small parts up took more than there is: from the part furthest above its share
        if (!change([&](int q) { return wgs[q] > 1; }, [&](int q) { return wgs[q] - wanted[q]; }, -1)) {
            if (lane == 0) atomicOr(&totals->refused, 1);
            return;
        }
    for (; used < nk; ++used)  // what rounding down left over goes where most is missing
        if (!change([&](int q) { return f[q + 1] - f[q] > wgs[q]; }, [&](int q) { return wanted[q] - wgs[q]; }, 1)) break;
    int mine = 0;
    for (int q = q0; q < q1; ++q) mine += wgs[q];
    int b = k * nk + wave_scan(mine) - mine;
    for (int q = q0; q < q1; ++q) {
        base[q] = b;
        b += wgs[q];
    }
}

// wgStart[b] = the place in the order at which workgroup b's virtual rows begin, for b in [0, budget]
__global__ __launch_bounds__(kBlock) void wg_starts_kernel(Parts P, int budget, const unsigned short *__restrict__ partOf, const int *__restrict__ length,
                                                           const int *__restrict__ first, const int *__restrict__ run, const int *__restrict__ partWgs,
                                                           const int *__restrict__ partBase, const Totals *__restrict__ totals, int *__restrict__ wgStart)
{
    const int i = blockIdx.x * kBlock + threadIdx.x;
    if (i > P.nV || totals->refused) return;
    auto workgroup = [&](int at) {
        const int p = partOf[at], f = first[p], rows = first[p + 1] - f, w = partWgs[p], seen = at - f;
        const long long entries = (long long)run[first[p + 1]] - run[f], before = (long long)run[at] - run[f];
        // (at least one virtual row per workgroup: the j-th starts no later than at the part's (rows - w + j)-th
        // virtual row and no earlier than at its j-th)
        int j = entries > 0 ? (int)(((before + length[at] / 2) * w) / entries) : 0;
        j = min(min(j, w - 1), seen);
        j = max(j, w - (rows - seen));
        return partBase[p] + j;
    };
    const int b = i < P.nV ? workgroup(i) : budget;
    for (int k = i > 0 ? workgroup(i - 1) + 1 : 0; k <= b; ++k) wgStart[k] = i;
}

// The virtual rows of workgroup blockIdx.x by length, longest first, those of one length in the order of the rows; chunkLen[b][i] = the longest of chunk i
__global__ __launch_bounds__(mxd::kThreads) void wg_order_kernel(Parts P, const int *__restrict__ wgStart, const int *__restrict__ order,
                                                                 const int *__restrict__ length, int bits, Totals *__restrict__ totals,
                                                                 int *__restrict__ sorted, int *__restrict__ chunkLen)
{
    using namespace mxd;
    __shared__ Digits digits;
    __shared__ int start[kDigits], part[kWaves];
    if (totals->refused) return;
    const int b = blockIdx.x, tid = threadIdx.x, lane = tid & 63, w = tid >> 6, i0 = wgStart[b], size = wgStart[b + 1] - i0;
    if (size == 0) return;
    if (size > kWgChunks * 64) {  // (its targets would not fit the LDS of the product)
        if (tid == 0) atomicOr(&totals->crowded, 1);
        return;
    }
    int d[kPer], at[kPer];
#pragma unroll
    for (int j = 0; j < kPer; ++j) d[j] = P.cap - length[i0 + min(w * kWave + j * 64 + lane, size - 1)];
    place_by_digit<true>([&](int j) { return d[j]; }, size, bits, digits, start, part, at);
#pragma unroll
    for (int j = 0; j < kPer; ++j) {
        const int i = w * kWave + j * 64 + lane;
        if (i >= size) continue;
        sorted[i0 + at[j]] = order[i0 + i];
        if (at[j] % 64 == 0) chunkLen[(size_t)b * kWgChunks + at[j] / 64] = P.cap - d[j];
    }
}

// Of every workgroup: its first chunk, its slice, the groups of rows that it counts off -- those of its rows, stretched so that
// the workgroups of a part cover all groups of the XCD between them.
__global__ __launch_bounds__(1024) void wg_groups_kernel(Parts P, int budget, const int *__restrict__ wgStart, const int *__restrict__ order,
                                                         const int *__restrict__ first, const int *__restrict__ partWgs, const int *__restrict__ partBase,
                                                         Totals *__restrict__ totals, int *__restrict__ wgSlice, int *__restrict__ wgChunk,
                                                         int *__restrict__ wgGroups)
{
    __shared__ int part[mxd::kWaves];
    const int tid = threadIdx.x, per = (budget + 1023) / 1024, b0 = min(budget, tid * per), b1 = min(budget, b0 + per);
    const bool dead = totals->refused || totals->crowded;
    if (dead) {  // (totals->nWG is zero: nothing is dealt)
        if (tid == 0) totals->refused = 1;
        return;
    }
    auto holds = [&](int b) { return wgStart[b + 1] - wgStart[b]; };
    int mine = 0, widest = 0;
    for (int b = b0; b < b1; ++b) mine += (holds(b) + 63) / 64;
    int at = mxd::sum_before(mine, part);
    for (int b = b0; b < b1; ++b) {
        const int k = b / P.nk;
        const int *f = first + (size_t)k * P.S;
        wgChunk[b] = at;
        at += (holds(b) + 63) / 64;
        int q = 0, ga = P.xg[k], n = 0;
        if (holds(b) == 0) {  // nothing to stream, no group to count off
            while (q < P.S - 1 && f[q + 1] == f[q]) ++q;
        } else {
            const int *base = partBase + (size_t)k * P.S, *wgs = partWgs + (size_t)k * P.S;
            while (!(b >= base[q] && b < base[q] + wgs[q])) ++q;
            int before = b - 1, next = b + 1;
            while (before >= base[q] && holds(before) == 0) --before;
            while (next < base[q] + wgs[q] && holds(next) == 0) ++next;
            auto group = [&](int i) { return P.vRow[order[i]] / GR; };
            if (before >= base[q]) ga = group(wgStart[b]);
            const int gb = next == base[q] + wgs[q] ? P.xg[k + 1] - 1 : max(group(wgStart[b + 1] - 1), group(wgStart[next]) - 1);
            n = gb - ga + 1;
        }
        wgSlice[b] = q;
        wgGroups[2 * (size_t)b] = ga;
        wgGroups[2 * (size_t)b + 1] = n;
        widest = max(widest, n);
    }
    const bool wide = __syncthreads_or(widest > mx::kFusedWgGroups);  // (a lane per group counts it off)
    if (widest > 0) atomicMax(&totals->maxWgGroups, widest);
    if (tid == 1023) {
        totals->nWG = wide ? 0 : budget;
        totals->chunks = wide ? 0 : at;
        if (wide) totals->refused = 1;
        wgGroups[2 * (size_t)budget] = wgGroups[2 * (size_t)budget + 1] = 0;
    }
}
__global__ __launch_bounds__(64) void wg_chunks_kernel(const Totals *__restrict__ totals, const int *__restrict__ wgStart, const int *__restrict__ wgChunk,
                                                       const int *__restrict__ chunkLen, int *__restrict__ list, int *__restrict__ first,
                                                       int *__restrict__ number, int *__restrict__ steps)
{
    const int b = blockIdx.x;
    if (b >= totals->nWG) return;
    const int c0 = wgChunk[b], i0 = wgStart[b], n = wgStart[b + 1] - i0;
    for (int i = threadIdx.x; i * 64 < n; i += 64) {
        list[c0 + i] = c0 + i;
        first[c0 + i] = i0 + 64 * i;
        number[c0 + i] = min(64, n - 64 * i);
        steps[c0 + i] = chunkLen[(size_t)b * kWgChunks + i];
    }
}
__global__ __launch_bounds__(64) void group_need_kernel(const int *__restrict__ wgGroups, int *__restrict__ groupNeed)
{
    const int g0 = wgGroups[2 * blockIdx.x], n = wgGroups[2 * blockIdx.x + 1];
    for (int i = threadIdx.x; i < n; i += 64) atomicAdd(&groupNeed[g0 + i], 1);
}
// target[place of virtual row t]: the k-th virtual row of row r at ((r / GR) * places + k) * GR + r % GR
__global__ __launch_bounds__(kBlock) void fused_targets_kernel(const int *__restrict__ segPtr, const int *__restrict__ segIdx, const int *__restrict__ vRow,
                                                               int nV, int places, int *__restrict__ target)
{
    const int t = blockIdx.x * kBlock + threadIdx.x;
    if (t >= nV) return;
    const int r = vRow[t];
    target[segIdx[t]] = (int)(((size_t)(r / GR) * places + (t - segPtr[r])) * GR + r % GR);
}
// the padding lanes of a chunk put theirs at the spare places behind the last group; 64 spare entries, zero
__global__ __launch_bounds__(kBlock) void spare_targets_kernel(int n, int spare, int *__restrict__ target)
{
    const int i = blockIdx.x * kBlock + threadIdx.x;
    if (i < n + 64) target[i] = i < n ? spare + (i & 63) : 0;
}

constexpr int kVrowsLeast = 16384;
bool fused_plan_on_device(int S, int cap, int nV) { return X * S <= mxd::kDigits && cap < mxd::kDigits && nV >= kVrowsLeast; }

int plan_fused_device(mx_dtype dtype, int budget, int S, int rows, int nnz, int cap, int nV, int mode, const int *rowPtr, const int *segPtr,
                      const int *vRow, const int *vSlice, const int *vLen, int *sorted, ChunkPlan &P, FusedPlan &F, bool *taken, hipStream_t s)
{
    const int nGroups = (rows + GR - 1) / GR, SPB = mx::kSliceBatchEntries / mx::slice_step_entries(dtype);
    *taken = false;
    if ((long long)nGroups * mx::kSliceLightSegs * GR > 2000000000LL || budget < X || budget % X || nGroups < X || nnz == 0) return MX_OK;
    const int n = X * S, tiles = (int)(((long long)nV + mxd::kTile - 1) / mxd::kTile);
    auto bits_of = [](int values) {
        int b = 0;
        while ((1 << b) < values) ++b;
        return b;
    };
    size_t scanBytes = 0;
    MXL_TRY(rocprim::exclusive_scan(nullptr, scanBytes, (const int *)nullptr, (int *)nullptr, 0, (size_t)nV + 1, rocprim::plus<int>(), s));
    Dealing D;
    const size_t v1 = (size_t)nV + 1, N = (size_t)nV / 64 + (size_t)budget;
    int rc = D.make(N, (size_t)budget, D.al((size_t)tiles * n * 4) + 5 * D.al((size_t)(n + 1) * 4) + D.al((X + 1) * 4) + 3 * D.al(v1 * 4) + D.al(v1 * 2) +
                                           D.al((size_t)n * 8) + D.al((size_t)(budget + 1) * 4) + D.al((size_t)budget * kWgChunks * 4) + D.al(scanBytes), P);
    if (rc) return rc;
    int *count = D.part<int>((size_t)tiles * n), *total = D.part<int>(n + 1), *first = D.part<int>(n + 1), *partWgs = D.part<int>(n + 1),
        *partBase = D.part<int>(n + 1), *flag = D.part<int>(n + 1);
    int *order = D.part<int>(v1), *length = D.part<int>(v1), *run = D.part<int>(v1);
    unsigned short *partOf = D.part<unsigned short>(v1);
    double *want = D.part<double>(n);
    int *wgStart = D.part<int>(budget + 1), *chunkLen = D.part<int>((size_t)budget * kWgChunks);
    Parts parts{S, rows, nGroups, budget / X, nV, cap, vRow, vSlice, vLen, D.part<int>(X + 1)};
    void *scanTmp = D.part<char>(scanBytes);
    MXL_TRY(mx::dev_malloc(&F.wgGroups.p, ((size_t)budget * 2 + 2) * 4));
    MXL_TRY(hipMemsetAsync(D.totals, 0, sizeof(Totals), s));
    MXL_TRY(hipMemsetAsync(length + nV, 0, 4, s));
    const Totals *T = D.totals;
    hipLaunchKernelGGL(most_vrows_kernel, dim3((unsigned)std::min(1024, (rows + kBlock - 1) / kBlock)), dim3(kBlock), 0, s, segPtr, rows, D.totals);
    hipLaunchKernelGGL(xcd_groups_kernel, dim3(1), dim3(64), 0, s, rowPtr, (long long)nnz, parts, D.totals);
    hipLaunchKernelGGL(part_counts_kernel, mxd::tile_blocks(tiles), dim3(mxd::kThreads), 0, s, parts, tiles, count);
    hipLaunchKernelGGL(mxd::bucket_offsets_kernel, dim3((unsigned)((n + 15) / 16)), dim3(1024), 0, s, count, n, tiles, total);
    hipLaunchKernelGGL(mxd::bucket_starts_kernel<false>, dim3(1), dim3(mxd::kThreads), 0, s, (const int *)total, n, mxd::BucketBound{}, (const int *)nullptr, 0, first, flag);
    hipLaunchKernelGGL(part_order_kernel, mxd::tile_blocks(tiles), dim3(mxd::kThreads), 0, s, parts, bits_of(n), tiles, (const int *)count, (const int *)first, order,
                       length, partOf);
    MXL_TRY(hipGetLastError());
    MXL_TRY(rocprim::exclusive_scan(scanTmp, scanBytes, (const int *)length, run, 0, v1, rocprim::plus<int>(), s));
    hipLaunchKernelGGL(part_shares_kernel, dim3(X), dim3(64), 0, s, parts, (const int *)first, (const int *)run, want, partWgs, partBase, D.totals);
    hipLaunchKernelGGL(wg_starts_kernel, grid((long long)nV + 1), dim3(kBlock), 0, s, parts, budget, (const unsigned short *)partOf, (const int *)length,
                       (const int *)first, (const int *)run, (const int *)partWgs, (const int *)partBase, T, wgStart);
    hipLaunchKernelGGL(wg_order_kernel, dim3((unsigned)budget), dim3(mxd::kThreads), 0, s, parts, (const int *)wgStart, (const int *)order, (const int *)length,
                       bits_of(cap), D.totals, sorted, chunkLen);
    hipLaunchKernelGGL(wg_groups_kernel, dim3(1), dim3(1024), 0, s, parts, budget, (const int *)wgStart, (const int *)order, (const int *)first,
                       (const int *)partWgs, (const int *)partBase, D.totals, D.wgSlice, D.wgChunk, F.wgGroups.as<int>());
    hipLaunchKernelGGL(wg_chunks_kernel, dim3((unsigned)budget), dim3(64), 0, s, T, (const int *)wgStart, (const int *)D.wgChunk, (const int *)chunkLen, D.list,
                       D.first, D.number, D.steps);
    MXL_TRY(hipGetLastError());
    if ((rc = D.deal(SPB, s))) return rc;
    // the slowest workgroup reads the sums of every group it covers after its last chunk: beyond kFusedAddBytes
    // of them that tail outweighs the launch saved, and the form is left unless it was asked for
    const int places = std::max(D.got.most, 1);
    const long long addBytes = (long long)D.got.maxWgGroups * places * GR * (dtype == MX_F64 ? 8 : 4);
    if (D.got.refused || (mode != 1 && addBytes > mx::kFusedAddBytes)) return MX_OK;
    if ((rc = D.emit(SPB, P, s))) return rc;
    MXL_TRY(mx::dev_malloc(&F.groupNeed.p, ((size_t)nGroups + 1) * 4));
    MXL_TRY(hipMemsetAsync(F.groupNeed.p, 0, ((size_t)nGroups + 1) * 4, s));
    hipLaunchKernelGGL(group_need_kernel, dim3((unsigned)budget), dim3(64), 0, s, F.wgGroups.as<int>(), F.groupNeed.as<int>());
    MXL_TRY(hipGetLastError());
    F.nGroups = nGroups;
    F.maxWgGroups = D.got.maxWgGroups;
    F.places = places;
    *taken = true;
    return MX_OK;
}

int fused_targets_device(int nGroups, int places, long long totalChunks, const int *segPtr, const int *segIdx, const int *vRow, int nV, int *target,
                         hipStream_t s)
{
    hipLaunchKernelGGL(spare_targets_kernel, grid(totalChunks * 64 + 64), dim3(kBlock), 0, s, (int)(totalChunks * 64), (int)((size_t)nGroups * places * GR), target);
    hipLaunchKernelGGL(fused_targets_kernel, grid(nV), dim3(kBlock), 0, s, segPtr, segIdx, vRow, nV, places, target);
    MXL_TRY(hipGetLastError());
    return MX_OK;
}

}  // namespace mxl

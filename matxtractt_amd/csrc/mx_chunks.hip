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

int plan_chunks_device(mx_dtype dtype, int budget, int S, int nV, const unsigned *sortedKey, unsigned perSlice, const int *sorted,
                       const int *vLen, ChunkPlan &P, hipStream_t s)
{
    const int E = mx::slice_step_entries(dtype), SPB = mx::kSliceBatchEntries / E;
    const long long chunksMost = (long long)nV / 64 + S;
    const size_t N = (size_t)chunksMost, G = (size_t)budget + 2 * (size_t)S + (size_t)(chunksMost / mx::kSliceWgChunks) + 1;
    auto al = [](size_t b) { return (b + 255) & ~(size_t)255; };
    // (one block of scratch, and one that the caller reads the chunks' facts from)
    const size_t sB = al(((size_t)S + 1) * 8), nB = al(N * 4 + 4), gB = al((G + 1) * 8);
    Buf scratch;
    MXL_TRY(mx::dev_malloc(&scratch.p, 6 * sB + 6 * nB + al(3 * N * 4 + 12) + 4 * gB + al(3 * G * 4) + al(G * W * 16) + 256));
    MXL_TRY(mx::dev_malloc(&P.made.p, 4 * nB + 2 * nB));
    unsigned char *b = (unsigned char *)scratch.p;
    auto part = [&](size_t bytes) {
        unsigned char *q = b;
        b += bytes;
        return (void *)q;
    };
    int *sliceStart = (int *)part(sB), *chunkBase = (int *)part(sB), *wgBase = (int *)part(sB);
    unsigned long long *work = (unsigned long long *)part(sB);
    double *missing = (double *)part(sB);
    int *groups = (int *)part(sB);
    int *first = (int *)part(nB), *number = (int *)part(nB), *steps = (int *)part(nB), *whose = (int *)part(nB), *place = (int *)part(nB),
        *list = (int *)part(nB), *how = (int *)part(al(3 * N * 4 + 12));
    int *wgSlice = (int *)part(gB), *wgChunk = (int *)part(gB), *wgSteps = (int *)part(gB);
    int *wgChunks = wgSteps + (G + 1);  // (a gB is eight bytes a workgroup)
    long long *wgStep = (long long *)part(gB);
    int *bins = (int *)part(al(3 * G * 4)), *wave4 = (int *)part(al(G * W * 16));
    Totals *totals = (Totals *)part(256);
    b = (unsigned char *)P.made.p;
    int *chunkFirst = (int *)part(nB), *chunkN = (int *)part(nB), *chunkSteps = (int *)part(nB), *chunkAt = (int *)part(nB);
    long long *chunkStep0 = (long long *)part(2 * nB);
    int *chunkEndTmp = whose;  // (free once the workgroups are dealt)
    hipLaunchKernelGGL(slice_chunks_kernel, dim3(1), dim3(1024), 0, s, sortedKey, nV, S, perSlice, sliceStart, chunkBase, work);
    hipLaunchKernelGGL(chunk_steps_kernel, grid(chunksMost), dim3(kBlock), 0, s, (const int *)sliceStart, (const int *)chunkBase, S, sorted, vLen, first, number,
                       steps, work);
    hipLaunchKernelGGL(slice_shares_kernel, dim3(1), dim3(64), 0, s, (const unsigned long long *)work, (const int *)chunkBase, S, budget, missing, groups,
                       wgBase, totals);
    hipLaunchKernelGGL(deal_slices_kernel, dim3((unsigned)S), dim3(64), 0, s, (const int *)steps, (const int *)chunkBase, (const int *)wgBase, bins, whose, place,
                       wgSlice, wgChunk, list);
    hipLaunchKernelGGL(deal_waves_kernel, dim3((unsigned)G), dim3(64), 0, s, (const Totals *)totals, (const int *)wgChunk, (const int *)list, (const int *)first,
                       (const int *)number, (const int *)steps, SPB, how, chunkFirst, chunkN, chunkSteps, chunkEndTmp, chunkAt, wave4, wgSteps, wgChunks);
    hipLaunchKernelGGL(wg_steps_kernel, dim3(1), dim3(1024), 0, s, (const int *)wgSteps, (const int *)wgChunks, wgStep, totals);
    MXL_TRY(hipGetLastError());
    Totals got{};
    MXL_TRY(hipMemcpyAsync(&got, totals, sizeof(got), hipMemcpyDeviceToHost, s));
    MXL_TRY(hipStreamSynchronize(s));
    if (got.steps * 64 * E > 2000000000LL || got.chunks * 64 > 2000000000LL) {
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
    hipLaunchKernelGGL(emit_chunks_kernel, dim3((unsigned)P.nWG + 1), dim3(64), 0, s, P.nWG, SPB, (const int *)wgSlice, (const int *)wgChunk, (const int *)wgChunks,
                       (const long long *)wgStep, (const int *)wave4, (const int *)chunkEndTmp, (const int *)chunkAt, (int)P.totalChunks, P.wgDesc.as<int>(),
                       P.waveDesc.as<int>(), P.chunkEnd.as<int>(), chunkStep0);
    MXL_TRY(hipGetLastError());
    P.chunkFirst = chunkFirst;
    P.chunkN = chunkN;
    P.chunkSteps = chunkSteps;
    P.chunkStep0 = chunkStep0;
    return MX_OK;  // (the scratch goes back to the scope, whose next request is served in the order of the stream)
}

}  // namespace mxl

// Device-side views shared by the plan code and the kernel launchers.
#pragma once
#include <hip/hip_runtime_api.h>

#include "matxtract_hip.h"

namespace mx {

// ---- device memory (mx_util.cpp).  Making a plan takes and gives back a hundred arrays, and hipMalloc and hipFree
// of large ones cost more than the kernels that fill them (64 MB: 21 + 52 us in an idle process, several times that
// beside other allocations).  dev_malloc and dev_free stand in for them and keep what was given back:
//  * inside a MemScope -- one per entry point that works on a stream -- a freed block serves the thread's next
//    request at once, in the order of that stream, and becomes anybody's when the scope ends, after the stream has
//    been waited for;
//  * inside IdleFrees, which waits for the device first, it is anybody's at once (plans that are destroyed: their
//    streams are the callers'); where that wait is refused the block goes back by hipFree;
//  * elsewhere dev_free waits for the device, as hipFree does (an IdleFrees of its own).
// Idle blocks hold at most 1/128 of the device's memory whenever a scope or an IdleFrees ends, go back to the device after 64 of
// those in which nobody asked for them, all of them when an allocation fails, and on mx_release_memory.  What a thread has
// given back inside a scope holds at most 1/16, and goes back to the device as well when an allocation of its own fails.
hipError_t dev_malloc(void **out, size_t bytes);
hipError_t dev_free(void *p);
void release_idle_memory();
// hipMemcpy to the device from memory that a caller allocated as it liked: large copies go through pinned buffers that the host's cores
// fill while the device reads them (a partition of 4.2 million binary64 entries, 50 MB, made on the device: 3.4 ms with hipMemcpy, of them 0.5 in
// the look at the columns by one core, 2.2 so).  The buffers (16 MB) are kept until mx_release_memory; a thread that finds them
// in use copies by hipMemcpy.
hipError_t copy_up(void *dst, const void *src, size_t bytes);
void release_staging();
struct MemScope {
    explicit MemScope(hipStream_t s);
    ~MemScope();
    MemScope(const MemScope &) = delete;
    MemScope &operator=(const MemScope &) = delete;
};
struct IdleFrees {
    IdleFrees();
    ~IdleFrees();
    IdleFrees(const IdleFrees &) = delete;
    IdleFrees &operator=(const IdleFrees &) = delete;
};

// The next of the places p, p + stride, .. below n; n where there is none (p + stride may be more than an int holds).  A thread's own first of
// the places [p, n) is next_of(p, n, thread): its number on top of a p near n may be more than an int holds, too.
__host__ __device__ inline int next_of(int p, int n, int stride) { return n - p > stride ? p + stride : n; }
// Rows, columns and entries that the kernels which lay a matrix out can number: they reach past the last row or entry by fewer
// than this leaves.  (From device arrays a plan refuses more than that; from host arrays the host's layouts take it.)
inline bool forms_can_number(int rows, int cols, int nnz)
{
    constexpr int most = 2147483647 - 512;
    return rows <= most && cols <= most && nnz <= most;
}

// CSR matrix resident on the device, plus the row ranges of the CSR kernel's workgroups.
// col/val carry kCsrPad extra zero entries so that a wave's aligned 128-bit loads may overrun.
struct DeviceCsr {
    int rows = 0, cols = 0, nnz = 0;
    int *rowPtr = nullptr;    // [rows+1]
    int *col = nullptr;       // [nnz + kCsrPad], or nullptr when the 16-bit form below is used
    unsigned short *col16 = nullptr;  // [nnz + kCsrPad] column ids as offsets from colBase[workgroup]
    int *colBase = nullptr;           // [nBlocks] lowest column of each workgroup's entries
    void *val = nullptr;      // [nnz + kCsrPad]
    int *blockDesc = nullptr; // [nBlocks][4] {first row, end row, first entry, end entry} per workgroup
    int nBlocks = 0;
    int npt = 0;              // entries per lane per tile the rows were packed for
    bool scan = false;        // sum the rows of a tile by a segmented scan (row lengths vary a lot)
    // a matrix with at most 256 distinct values (a stencil, a graph): one byte per entry that
    // names the value, and the values themselves (padded to 256); used with col16 only
    unsigned char *codes = nullptr;  // [nnz + kCsrPad]
    void *dict = nullptr;            // [256]
    int nDict = 0;
    bool useDict = false;            // the plan found this form the faster one
};
constexpr int kCsrPad = 1088;  // a wave may read one whole wave tile (64*16 entries) past the end

// Entries per lane per tile of the CSR kernel (a tile is 256 lanes wide).
int csr_entries_per_lane(mx_dtype dtype);

// Tiles resident on the device, re-packed for the tile kernels.  The fragments the plan
// selects are expanded from the reference's encoding (bitmap + packed values) into full
// fragM x fragK blocks, zeros included (row-major inside a block), so that a lane can load
// exactly what the matrix core wants from it with no decoding; the plan only selects fragments
// that are mostly full.  The columns of a chunk's selected fragments are first put in ascending
// order of the caller's column ids and cut into blocks anew (the reference orders them by their
// rank among the dense columns, which scatters neighbours): gathers touch fewer lines, and dense
// strips become blocks of consecutive columns.  (Rows of binary16 strips do not come from the
// reference's chunks at all: the plan groups them into chunks of its own, see `dense`.)  The
// blocks are grouped into "steps" -- what one wave feeds to the matrix core at a time: two
// halves of up to tile_slots(dtype)/2 blocks.  A chunk with more
// selected fragments than half a step takes whole steps of its own (filling half 0 first; its
// two halves are added at the end); smaller chunks share a step, one per half.  Per step:
//   hdr    kTileHdr dwords: [0,16) output row of each of the 8 rows of half 0 and half 1
//          (-1 = none); [16] flags (1 = store the sums after this step, 2 = the halves are
//          different chunks); [17],[18] blocks in half 0 and half 1; [19],[20] first value
//          and blocks in half 0 of the step four further on (a wave learns where to prefetch
//          from there; its own last step when it has no such step); [21,29) first column of
//          the block in each slot (-1 = none), used by the strip form of the binary16 kernel.
//   atox   64 column ids (slot-major), -1 for unused ones
//   values the blocks of half 0, then those of half 1; nothing for absent blocks.
// Waves take whole chunks: waveDesc = {first step, end step, first value of the wave's first
// four steps, blocks in half 0 of each of them (one byte each), 0}.
struct DeviceTiles {
    int chunkNum = 0;  // chunks with at least one selected fragment
    int frags = 0, vals = 0;   // selected fragments, entries they hold
    long long stored = 0;      // values stored (zeros included)
    int steps = 0, nWaves = 0;
    bool dense = false;        // binary16 chunks the plan formed from rows of dense strips: every block's eight
                               // columns are consecutive and every chunk fits one step
                               // (two share a step when both fit a half): tile_dense_kernel can run it
    bool ownedRows = false;    // set by the plan: no row of these tiles gets anything from the CSR part
    // binary64 `dense` layouts (blocks of 8 x 8 on rows that the CSR part shares) when they ride in the
    // combine kernel's launch: per step 128 indices into the slice layout's sums -- half h, row i,
    // place j at [64h + 8i + j], -1 = none -- set on the step after which the half's sums are stored
    int *vidx = nullptr;
    int *waveDesc = nullptr;   // [nWaves][8]
    int *hdr = nullptr;        // [steps][kTileHdr]
    int *atox = nullptr;       // [steps][64]
    void *tcVal = nullptr;     // blocks
};
constexpr int kTileHdr = 32;
inline int tile_slots(mx_dtype d) { return d == MX_F64 ? 16 : 8; }  // fragment slots per step
// slot of block i of half h: binary64 MFMA j takes slots 2j and 2j+1, binary16 slots 0..3 and 4..7
inline int tile_slot(mx_dtype d, int half, int i) { return d == MX_F64 ? 2 * i + half : 4 * half + i; }

// The CSR part (or the rows of it that the plan selects) re-laid for x resident in LDS.  The
// columns are cut into S slices of sliceCols columns (a slice of x fits LDS).  The entries of
// a row that fall into one slice form a "virtual row"; one longer than the plan's cap is cut
// into several, so a matrix row owns one or more virtual rows and its result is the sum of
// theirs.  Per slice the virtual rows are sorted by length (among equals by the kind of their
// row -- sole virtual row, a few, many -- then by row) and cut into chunks of 64, one
// virtual row per lane (a sliced-ELL layout: every row of a chunk is padded to the chunk's
// longest, and the sort keeps that padding small).  A slice gets workgroups in proportion to
// its entries, its chunks are dealt to them longest first, and inside a workgroup to its waves
// the same way.  A lane walks its virtual row one entry -- one "step" -- at a time; a wave's
// chunks follow each other in the wave's stream, which is stored in batches of
// kSliceBatchEntries entries per lane
// (zero-padded to a whole batch at the end): per batch the lanes' column offsets (lanes
// contiguous), then their values -- binary16: lanes contiguous; binary64: one sub-block of 16
// bytes (two values) per lane -- so that every load of a wave is one contiguous stretch.
// Chunks are numbered workgroup by workgroup, wave by wave; virtual row v = 64 * chunk + lane
// puts its sum into partial[v], and a second kernel turns those into y: rowInfo[r] is the
// virtual row of a matrix row that owns exactly one, -1 for a row that owns none, -2 for a row
// that owns several.  Of those, the rows with up to kSliceLightSegs virtual rows are lightRow[i]
// with their virtual rows in lightIdx[i][kSliceLightSegs] (-1 = none); the rows with more are
// heavyInfo[i] = {row, first index into segIdx, count, 0} with their virtual rows listed in
// segIdx.
struct DeviceSlices {
    int nWG = 0, S = 0, rows = 0, cols = 0, sliceCols = 0;
    int maxWgChunks = 0;              // chunks of the largest workgroup (their ends are kept in LDS)
    long long steps = 0;              // total steps stored (64 lanes, one entry each)
    long long chunks = 0;             // total chunks
    int nnz = 0;                      // entries held
    int vrows = 0;                    // virtual rows
    bool subset = false;              // only some rows are held: their sums are added to y, the others left alone
    int *wgDesc = nullptr;            // [nWG][4] {slice, first chunk, chunks, 0}
    int *waveDesc = nullptr;          // [nWG*kSliceWaves][4] {first batch, batches, first chunk inside the workgroup, chunks}
    int *chunkEnd = nullptr;          // [chunks] step, counted from the wave's first, at which the chunk ends
    unsigned short *ecol = nullptr;   // [batches][64][kSliceBatchEntries] col - slice * sliceCols
    void *eval = nullptr;             // [batches] values, laid out as described above
    // a matrix with at most 256 distinct values: a byte per entry (at the place of its column
    // offset) that names the value, and the values (padded to 256)
    unsigned char *ecode = nullptr;   // [batches][64][kSliceBatchEntries]
    void *dict = nullptr;             // [256]
    int nDict = 0;
    bool useDict = false;             // the plan found this form the faster one
    void *partial = nullptr;          // [chunks*64] accumulators
    int *rowInfo = nullptr;           // [rows, padded to a multiple of 4 with -2]
    int *segIdx = nullptr;            // [vrows] virtual rows listed matrix row by matrix row
    int *lightRow = nullptr;          // [nLight]
    int *lightIdx = nullptr;          // [nLight][4 * lightQuads]
    int lightQuads = 2;               // 1 when no light row has more than four virtual rows
    int *heavyInfo = nullptr;         // [nHeavy][4]
    int nLight = 0, nHeavy = 0;
    int mostVrows = 0;                // most virtual rows of any row
    bool keep = false;                // the entries are read with plain loads (they may stay in the caches), not streamed
    // The one-launch form (csr_slice_kernel<.., FUSED>), when the layout was made for it: the rows are cut
    // into groups of kFusedGroupRows, the groups into one contiguous range per XCD, and the virtual rows
    // of a slice are ordered by group before length, so that a workgroup's chunks cover a contiguous run
    // of groups.  Logical workgroups [k * nWG / 8, (k + 1) * nWG / 8) belong to XCD k, and a workgroup of
    // the launch that runs on XCD k takes one of those (which one: blockIdx / 8), so all workgroups that
    // hold sums of a group share an L2: they store their sums with plain stores, which meet there,
    // count themselves off on the group's counter with an atomic that executes there, and the one that
    // completes the count adds the sums of the group's rows up and writes y.  Nobody waits.  The sums do
    // not go to `partial` in this form but to fusedSums, laid out for the one who adds: the k-th
    // virtual row of row r at [((r / G) * placesPerRow + k) * G + r % G], G = kFusedGroupRows, so that a
    // wave that adds 64 consecutive rows reads 64 consecutive sums per place and needs no index list;
    // fusedTarget names that place for every virtual row (a workgroup keeps its chunks' part of it in
    // LDS, which bounds the chunks a workgroup may have).  A place that no virtual row owns keeps the zero
    // it was allocated with, so the one who adds takes all placesPerRow places of a row without asking how
    // many count.  The arrays above stay valid for the two-launch form, which a plan falls back to.
    bool fused = false;
    int nGroups = 0, maxWgGroups = 0;
    int placesPerRow = 0;             // most virtual rows of a row (1 .. 8)
    int *wgGroups = nullptr;          // [nWG][2] {first group, groups} whose counters the workgroup bumps
    int *groupNeed = nullptr;         // [nGroups] workgroups that bump the group's counter
    int *groupCount = nullptr;        // [nGroups] the counters; zero between launches (the last arriver clears its own)
    int *fusedTarget = nullptr;       // [chunks * 64] where virtual row 64 * chunk + lane puts its sum (a spare place for padding lanes)
    void *fusedSums = nullptr;        // [nGroups * placesPerRow * G + 64] accumulators; zero where no virtual row writes
    unsigned *claim = nullptr;        // [nWG] launches in which each logical workgroup's work was taken (once each)
};
constexpr int kFusedGroupRows = 256;  // rows whose sums one arriver adds up at a time
constexpr int kFusedXcds = 8;         // L2 domains of the device the one-launch form is laid out for
constexpr int kFusedWgChunks = 96;    // most chunks of a workgroup in that form (their targets, 256 bytes each, share the LDS with x)
constexpr int kFusedWgGroups = 255;  // most groups a workgroup may hold sums of
constexpr int kFusedAddBytes = 100 * 1024;  // most bytes of sums under one workgroup (groups x places x a group's rows) for which
                                            // the form is taken unasked: the slowest workgroup of a launch reads that much after its last
                                            // chunk (about 70 ns per 2 KB), and beyond this a second launch is the faster way
constexpr int kFusedSlicesMost = 8;          // ... and most slices: every XCD copies every slice of x in this form (a slice's workgroups are
                                            // spread over all eight), 64 ns a slice more than when one XCD has a slice to itself
constexpr long long kKeepL2Bytes = 24LL << 20;      // entries of a slice layout up to this size fit the eight L2s beside x and the sums
constexpr long long kKeepCacheBytes = 192LL << 20;  // ... and up to this size the memory-side cache beside everything else a product touches
constexpr long long kKeepHandoffBytes = 10LL << 20;  // what the second launch must move per product (sums, row tables, y) to push streamed
                                                    // entries out of the memory-side cache fast enough for plain loads to pay
constexpr int kSliceBytes = 131072;   // the slice of x a workgroup keeps in LDS
constexpr int kSliceLdsMax = 163840;  // LDS of a CU
constexpr int kSliceWgChunks = 4096;  // most chunks a workgroup may have
constexpr int kSliceWaves = 8;        // waves per workgroup; one workgroup per CU
constexpr int kSliceThreads = 64 * kSliceWaves;
inline int slice_cols(mx_dtype d) { return kSliceBytes / (d == MX_F64 ? 8 : 2); }
constexpr int kSliceBatchEntries = 8;  // entries a lane loads at a time
constexpr int kSliceChunkCost = 2;     // what ending a chunk costs a wave, in steps of its stream (for dealing chunks out evenly)
inline int slice_step_entries(mx_dtype) { return 1; }  // entries a lane takes per step; chunks end between steps
constexpr int kSliceLightSegs = 8;     // rows with at most this many virtual rows are summed by one lane

// The CSR part of a matrix whose rows repeat a pattern of column offsets (a stencil, a few diagonals):
// chunks of 64 * R consecutive rows (R = 2 binary64, 4 binary16), each of them one to four waves' (offsets_waves), with the ascending
// list of the offsets (column - row) that its rows have.  Per chunk and unit -- unitBytes per lane, one
// contiguous stretch per wave -- the values of U offsets for the R rows of every lane; a place that no
// entry owns holds -0.0 (any binary64 whose upper half is 0x80000000) or code 255.
struct DeviceOffsets {
    int rows = 0, cols = 0, nnz = 0, nChunks = 0;
    int units = 0, unitBytes = 0;  // units of all chunks; bytes per lane and unit (16 of values, 8 of codes)
    long long nOffs = 0;
    int *chunk = nullptr;    // [nChunks][4] {first unit, first offset, units, flags: 1 = reaches outside x, 2 = reaches past the last row}
    int *offs = nullptr;     // [nOffs] U per unit, the last of a chunk repeated up to whole units
    void *stream = nullptr;  // [units][64] unitBytes each
    void *dict = nullptr;    // [256] values, when the units hold codes
    int nDict = 0;
    bool keep = false;       // the units are read with plain loads (they may stay in the caches), not streamed
};
constexpr int kOffsetsMost = 64;           // most offsets of a chunk
constexpr int kOffsetsRowsLeast = 1024;    // fewest rows of a matrix that takes the form (2431 rows: 3.3 us, row tiles 3.3)
// A chunk's list of more than 40 offsets (binary16: 48) is two rounds of its four waves, one after the other, and a small matrix has
// nothing else to do meanwhile: 1100 rows of 60, binary64, 4.3 us, row tiles 3.1; 5000 4.4, 3.4; 10 thousand 4.4, 3.9; 20 thousand 4.4, 5.0; of 48, 5000
// 3.8, 3.4; 10 thousand 3.8, 3.6; 20 thousand 3.9, 4.6; of 40, 3000 3.5, 3.4; 10 thousand 3.5, 3.8; binary16, of 60, 5000 4.7, 4.0; 10
// thousand 4.7, 4.3; 20 thousand 4.7, 4.6; of 48, 5000 4.0, 4.3.  With one byte per binary64 value the second round is half as long
// (5000 rows of 60: 3.6, 3.6).
inline bool offsets_lists_pay(bool f64, bool dict, int longest, int nnz)
{
    if (f64 && dict) return true;
    return longest <= (f64 ? 40 : 48) || nnz >= (f64 ? 700000 : 1300000);
}
inline bool offsets_size_ok(int rows, int cols, int nnz)
{
    return forms_can_number(rows, cols, nnz) && rows >= kOffsetsRowsLeast && nnz >= rows && (long long)nnz <= (long long)rows * kOffsetsMost;
}
constexpr int offsets_chunk_rows(bool f64) { return f64 ? 128 : 256; }
constexpr double kOffsetsFill = 1.2;       // most places per entry: 9.6 bytes per binary64 entry, as much as with a column offset of two bytes
// What a product may touch for its units to be read with plain loads.  Plain / streaming loads, us, back to back | three
// plans in turn: 67 MB 11.9 / 12.2 | 11.8 / 13.1; 98 MB 15.6 / 16.7 | 17.4 / 17.6; 142 MB 21.3 / 23.0 | 28.8 / 25.1;
// 166 MB 24.2 / 26.8 | 32.3 / 28.7: from half of the memory-side cache on, anything else a program touches costs more
// than staying there gives.
constexpr long long kOffsetsKeepBytes = 128LL << 20;
constexpr int offsets_unit_bytes(bool dict) { return dict ? 8 : 16; }
// Waves that share a chunk.  Four: a wave's trips to memory are fewer and more of them are in flight on a matrix of few chunks
// (one / two / four waves, us, binary64, 27 offsets: 22 thousand rows 6.3 / 4.2 / 3.2; 717 thousand 33.1 / 31.2 / 28.6; 1.2 million
// 52.9 / 51.3 / 48.3).  One where a chunk's list is a single round of a wave: the others would have nothing to ask for, and the
// workgroups, which start at about one a nanosecond, are four times as many (1.5 million rows, binary64: one offset 6.7 / 8.5 / 12.4, three 10.3
// / 11.6 / 17.0, eight 18.7 / 18.2 / 20.3, fourteen 35.8 / 32.7 / 30.9; binary16: two 3.7 / 4.1 / 5.5, eight 5.3 / 5.3 / 7.7; row tiles of the first two: 7.3, 14.4); with more
// than four offsets from the size on where the workgroups outweigh what four waves ask for sooner (four waves / one: binary16, eight offsets, 25 to 180 thousand rows 2.9 / 3.1 to
// 3.2, 240 thousand 3.1 / 3.3, 358 thousand 3.55 / 3.5, 717 thousand 4.8 / 3.8; binary64, 90 thousand 3.0 / 3.0, 120 thousand 3.3 / 3.1).
// With one byte per binary64 value the kernel is bound by what a wave computes and the sum of the parts costs more than
// it gives from about two thousand chunks on (290 thousand rows 6.5 / 6.1 / 6.4, 717 thousand 10.9 / 10.5 / 11.7, a million 13.1 / 13.7 / 14.8).
inline int offsets_waves(bool f64, bool dict, long long nOffs, int nChunks)
{
    if (nOffs <= (nChunks < 1024 ? 4ll : 8ll) * nChunks) return 1;
    return f64 && dict && nChunks >= 2048 ? 2 : 4;
}
// Workgroups of a product: four waves each.
inline int offsets_blocks(bool f64, const DeviceOffsets &D)
{
    const int chunks = 4 / offsets_waves(f64, D.nDict > 0, D.nOffs, D.nChunks);
    return (D.nChunks + chunks - 1) / chunks;
}
void free_offsets(DeviceOffsets &D);
// Lays the matrix out in this form if it suits it (D.nChunks > 0 then); otherwise D stays empty and MX_OK is returned.
// (weak: a host-only link of the library's C++ files has no device code to call)
__attribute__((weak)) int build_offsets_device(mx_dtype dtype, int rows, int cols, int nnz, const int *rowPtr_dev, const int *col_dev,
                                               const void *val_dev, DeviceOffsets &D, hipStream_t s);
__attribute__((weak)) hipError_t launch_offsets(mx_dtype dtype, const DeviceOffsets &D, const void *x, void *y, hipStream_t s);

// The CSR part of a matrix whose neighbouring rows reach into one stretch of x (a mesh numbered for a small bandwidth):
// chunks of 64 consecutive rows, a row per lane, kWindowWaves of them to a workgroup, which puts the window of x that its rows
// reach into LDS.  Per chunk and unit four entries of every row: their places in the window (16 bits) and their values; a
// place that no entry owns is zeroPlace, where the kernel puts a zero, with the value zero.  Entries outside the
// window are kept with their columns and gathered from memory.
struct DeviceWindows {
    int rows = 0, cols = 0, nnz = 0, nChunks = 0, nWG = 0;
    int units = 0, unitBytes = 0;      // units of all chunks; bytes of a wave's unit
    int zeroPlace = 0, ldsBytes = 0;   // elements of the widest window; LDS of a workgroup
    int *window = nullptr;             // [nWG][2] {first element of x, vectors of 16 bytes}
    int farSteps = 0;                  // of all chunks: a step is one entry outside the window per row
    int nApart = 0;                    // chunks that a workgroup of its own gathers from memory
    int *chunk = nullptr;              // [nChunks][4] {first unit, units (-1: a chunk apart), first far step, far steps}
    int *apart = nullptr;              // [nApart] chunks, ascending
    unsigned char *stream = nullptr;   // [units + 1][unitBytes]
    int *farCol = nullptr;             // [farSteps + 1][64] columns, -1 for none
    void *farVal = nullptr;            // [farSteps + 1][64] values
    bool keep = false;                 // the units are read with plain loads (they may stay in the caches), not streamed
};
constexpr int kWindowUnit = 4;                // entries of a row in a unit
constexpr int kWindowWaves = 8;               // chunks (and waves) of a workgroup
constexpr int kWindowRowsLeast = 32768;       // fewest rows of a matrix that takes the form (33 thousand of 40 entries, binary16: 4.3 us, row tiles 5.3)
constexpr int kWindowEntriesLeast = 600000;   // binary64: fewest entries (0.33 million: 4.0 us, row tiles 3.8; 0.9 million: 4.2, 4.7)
constexpr double kWindowFill = 1.5;           // most bytes stored per byte of the entries
constexpr int kWindowMeanLeast = 4;           // fewest entries a row on average
inline bool window_size_ok(bool f64, int rows, int cols, int nnz)
{
    return forms_can_number(rows, cols, nnz) && rows >= kWindowRowsLeast && cols >= 64 && (long long)nnz >= (long long)rows * kWindowMeanLeast && nnz <= 1500000000 &&
           !(f64 && nnz < kWindowEntriesLeast);
}
// What a product may touch for its units to be read with plain loads.  Plain / streaming loads, us, back to back | three plans in
// turn: binary16, 51 MB 11.3 / 12.0 | 11.2 / 12.6; 76 MB 14.2 / 14.2 | 14.2 / 14.9; 99 MB 16.7 / 16.2 | 18.6 / 17.2; 108 MB 18.9 / 21.7 | 23.1 /
// 22.7; 126 MB 19.5 / 19.1 | 23.3 / 20.3; binary64, 79 MB 14.7 / 15.7 | 14.8 / 16.7; 100 MB 16.5 / 17.6 | 18.4 / 18.6; 120 MB 18.8 / 19.2 | 23.3 / 20.0;
// 132 MB 20.5 / 21.2 | 25.1 / 22.6.  Beyond 110 MB that is a trade, and against the slices these matrices had before plain loads come out
// ahead (127 MB, binary16: 1.5 million rows of 16, plain 22.9 | 29.7, streaming 26.8 | 27.2, slices 25.1 | 29.6; 600 thousand of 40, 20.3 | 25.9,
// 23.4 | 24.3, 22.2 | 25.4).
constexpr long long kWindowKeepBytes = 128LL << 20;
// Estimated time of a product in this form, us: the launch, a wait for the window per round of workgroups over the CUs, and the stored
// bytes, which come from the L2s, the memory-side cache (`touched` bytes have to fit) or memory -- or what one workgroup's CU takes in, 45 to 80
// bytes a nanosecond, where there are few workgroups.  (Least squares over 647 bands of 33 thousand to 3.2 million rows of 4 to 300 entries, on
// average 7 % off in binary64, 8 in binary16.)
inline double window_estimate(bool f64, double stored, double touched, int nWG, int nCU)
{
    const double MB = stored * 1e-6, own = MB / nWG * 1e3, rounds = (nWG + nCU - 1) / nCU, beyond = std::max(0.0, MB - 30.0);  // (own: KB of a workgroup)
    if (touched <= (double)kWindowKeepBytes)
        return f64 ? std::max(2.22 - 0.00146 * nWG + 1.3 * rounds + 0.084 * MB + 0.049 * beyond, 2.2 + own / 78)
                   : std::max(2.06 - 0.00044 * nWG + 0.93 * rounds + 0.064 * MB + 0.109 * beyond, 2.2 + own / 58);
    return f64 ? std::max(-2.59 + 0.00669 * nWG + 0.156 * MB, 2.2 + own / 44) : std::max(-1.65 + 0.0032 * nWG + 0.159 * MB, 2.2 + own / 45);
}
// Whether a matrix laid out in `stored` bytes by nWG workgroups is better off in this form than in the one it would have otherwise, which
// takes `other` us (other_forms_us).  Of the 647 bands the form was more than 3 % slower than the one before it 100 times, at worst 2.2 times
// as slow (33 thousand rows of 150 to 450 entries, binary64, 65 workgroups: 43.7 us, slices 20.2; 600 thousand of 28 to 52: 55, 48; 1.5
// million of 6: 42, 29.5; 3.2 million of 9, binary16: 49, 33); where this takes it (508 of them), 5 times, by 0.25 us at most (80 thousand rows of 8, binary64:
// 4.0, row tiles 3.8).  Few workgroups with more than so many bytes each also fall behind once the matrix shares the caches with
// anything else (33 thousand rows of 300, binary64, 95 MB, three plans in turn: 31 us, slices 21), and in binary16 small matrices have the one-launch
// slices (33 thousand of 300: 11.8 to 14.8, 11.2 to 11.5).
inline bool window_form_pays(bool f64, int nnz, double stored, double touched, int nWG, int nCU, double other)
{
    if (stored > kWindowFill * (double)nnz * (f64 ? 10 : 4) + 65536) return false;
    const double most = f64 ? 0.8e6 : nWG * 8 < nCU * 3 ? 0.3e6 : 0.7e6;
    if (nWG * 16 < nCU * 15 && stored > most * nWG) return false;
    return window_estimate(f64, stored, touched, nWG, nCU) <= other;
}
// What the row tiles or the slices of a matrix take whose neighbouring rows reach into one stretch of x, by csr_estimates: the estimate of
// the one the plan would choose, brought to what these matrices were measured at (mx_plan.cpp).
double other_forms_us(mx_dtype dtype, int rows, int cols, int nnz, double linesPerGather);
constexpr double kWindowFarMost = 0.12;       // most entries outside the windows, of all
constexpr int kWindowFarSteps = 3;            // most entries of a row outside the window, but for chunks apart
constexpr int kWindowTrim = 32;               // bytes that a far entry is worth: an end of the window with fewer entries is left out
constexpr int kWindowLongest = 1024;          // most entries of a row
constexpr double kWindowShare = 0.6;          // most bytes of a window per byte of its workgroup's entries
constexpr int kWindowBytesMost = 80 << 10;    // of a window: two workgroups share the LDS of a CU
constexpr int kWindowBuckets = 2048;          // of columns, to find the windows with
// Elements of x in a window, at most: it costs its workgroup as much intake as entries do -- at most kWindowShare of their bytes, and what
// fits in LDS.
inline int window_widest(bool f64, int nnz, int nWG)
{
    const int es = f64 ? 8 : 2;
    return (int)std::min<double>(kWindowBytesMost, kWindowShare * ((double)nnz / nWG * (es + 2))) / es;
}
// Columns of a bucket, a multiple of a vector of x (cols >= 1; no sum here leaves the range of an int).
__host__ __device__ inline int window_bucket(int cols, int epv) { return ((cols - 1) / kWindowBuckets + epv) / epv * epv; }
// Whether a workgroup with `outside` of its n entries outside its window is one of a matrix of another kind.
__host__ __device__ inline bool window_scattered(int outside, int n) { return (long long)outside * 4 > (long long)n * 3 + 256; }
constexpr int window_unit_bytes(bool f64) { return 64 * kWindowUnit * (f64 ? 10 : 4); }
void free_windows(DeviceWindows &D);
// As build_offsets_device and launch_offsets.
__attribute__((weak)) int build_windows_device(mx_dtype dtype, int rows, int cols, int nnz, const int *rowPtr_dev, const int *col_dev,
                                               const void *val_dev, DeviceWindows &D, hipStream_t s);
__attribute__((weak)) hipError_t launch_windows(mx_dtype dtype, const DeviceWindows &D, const void *x, void *y, hipStream_t s);

// The sums of the virtual rows (DeviceSlices::partial) of mx_spmv_static live in a fixed array
// in device memory instead of the plan's own buffer: static_scratch gives the address of the
// current device's copy (looked up once per device, no allocation).
constexpr size_t kStaticScratchBytes = (size_t)32 << 20;  // the largest benchmark workload needs 27 MB
hipError_t static_scratch(void **ptr);

}  // namespace mx
#include <algorithm>
#include <vector>
namespace mx {
// One chunk of a slice on its way into the layout: `first` = index of its first virtual row in
// the sorted order of virtual rows, n = how many it has (64 but for the last of a slice), steps
// = the length of its longest (first) member.
struct SliceChunk {
    int first, n, steps;
};
// What plan_slice_chunks decides: the descriptors the kernels read (DeviceSlices) and, for every
// chunk in its final numbering (workgroup by workgroup, wave by wave), where it comes from and at
// which step of the streams it starts.
struct SlicePlan {
    int nWG = 0, maxWgChunks = 0;
    long long totalSteps = 0, totalChunks = 0;
    std::vector<int> wgDesc, waveDesc, chunkEnd;
    std::vector<int> chunkSlice, chunkFirst, chunkN, chunkSteps;
    std::vector<long long> chunkStep0;
    // one-launch form only
    int nGroups = 0, maxWgGroups = 0;
    std::vector<int> wgGroups, groupNeed;
};
int plan_slice_chunks(mx_dtype dtype, int budget, int S, const std::vector<std::vector<SliceChunk>> &sliceChunks, SlicePlan &P);
// The plan of the one-launch form from the records of the virtual rows (in the order of the rows, ascending
// columns inside a row: the numbering both layout routes use): `sorted` receives the order in which the
// virtual rows are laid out and P the workgroups, waves, chunks and groups.  `mode` 1: wherever the matrix
// suits the form; 2: only while the busiest workgroup has at most kFusedAddBytes of sums under it.  Returns 1
// when the form is taken (*places = places per row), 0 when it is not (nothing filled), a negative error code
// when the plan cannot be made (the error is set).
int plan_fused_records(mx_dtype dtype, int budget, int S, int rows, int cap, const int *rowPtr, const int *segPtr, const int *vSlice,
                       const int *vLen, int nV, int mode, std::vector<int> &sorted, SlicePlan &P, int *places);
// Where the virtual rows of the one-launch form put their sums (DeviceSlices::fusedTarget), from the places the
// layout gave them.
void fused_targets(int rows, int nGroups, int places, long long totalChunks, const int *segPtr, const int *segIdx, std::vector<int> &target);
constexpr int kSlicePadSteps = 16;  // spare zero steps after the last of the streams
// The slice layout built on the device from a CSR matrix in device memory (mx_layout.hip): the
// arrays of `D` equal those of the host route byte for byte.  `elsewhere_dev`: optional marks per
// row (device memory) as in the host route.  segPtrOut / segIdxOut (optional): host copies of the
// virtual rows of every row.  `fused` (1 or 2, as in plan_fused_records): the one-launch form where the matrix
// suits it (D.fused says whether it did); who plans it, the device or the host, fused_plan_on_device says.
int build_slices_device(mx_dtype dtype, int rows, int cols, int nnz, const int *rowPtr_dev, const int *col_dev, const void *val_dev,
                        int nCU, int S, const char *elsewhere_dev, DeviceSlices &D, hipStream_t s, std::vector<int> *segPtrOut = nullptr,
                        std::vector<int> *segIdxOut = nullptr, int fused = 0);

// The value dictionary of a matrix in device memory, as make_value_dict gives it on the host: at most `most`
// distinct bit patterns, numbered in the order of their first entry.  *codes = nnz bytes in device memory (the
// caller releases them; null when the matrix has more values), dict = 256 values in host memory, zero-padded.
int value_dict_device(mx_dtype dtype, const void *val_dev, int nnz, int most, void **codes, std::vector<unsigned char> &dict, int *nDict,
                      hipStream_t s);

// For plans made from a matrix that lives in device memory: the caller's arrays looked at before
// they are used as addresses; the mean number of distinct lines of x per wave-wide gather (sampled
// as on the host; launch_lines_per_gather adds the lines of at most some 2 * `most` sampled windows to *sum and waits for
// nothing); the row-tile form from device arrays (`desc` = pack_rows of the row pointers).
int check_csr_device(int rows, int cols, int nnz, const int *rowPtr_dev, const int *col_dev, hipStream_t s, const char *who);
int lines_per_gather_device(mx_dtype dtype, int nnz, const int *col_dev, hipStream_t s, double *out);
hipError_t launch_lines_per_gather(mx_dtype dtype, int nnz, const int *col_dev, int most, unsigned long long *sum, long long *sampled, hipStream_t s);
int upload_csr_device(mx_dtype dtype, int rows, int cols, int nnz, const int *rowPtr_dev, const int *col_dev, const void *val_dev,
                      const std::vector<int> &desc, bool scan, DeviceCsr &A, hipStream_t s);

// The host half of a hybrid plan done on the device (mx_hybrid.hip), for a matrix that lives in
// device memory.  analyse() runs the extraction and counts what the plan's decision needs;
// csr_part() assembles the CSR part (residual rows, then the entries of A_dd that stay) in the
// caller's numbering, in new device arrays that pass to the caller; strip_layout() lays the
// binary16 strip chunks out as steps (the caller plans the steps from the chunks' block counts,
// as the host route does).  All arrays equal the host route's byte for byte.
// The device arrays of a partition that was made on the device (mx_partition::twin): the two orders, A_dd and
// the residual, the tile encoding.  HybridDevice::adopt plans from them without any copy.
struct PartitionTwin {
    mx_dtype dtype = MX_F64;
    int rows = 0, cols = 0, nnz = 0, dRows = 0, dCols = 0, nDD = 0, nCD = 0;
    void *order = nullptr;  // descColId [cols], descRowId [rows] (its first dRows are rId)
    int *dc = nullptr, *dr = nullptr;
    void *split = nullptr;  // ddRowPtr, ddColInd, ddVal, cdRowPtr, cdColInd, cdVal
    int *ddp = nullptr, *ddc = nullptr, *cdp = nullptr, *cdc = nullptr;
    void *ddv = nullptr, *cdv = nullptr;
    mx_device_tiles T{};
};

struct HybridCounts {
    long long generalFrags = 0, generalEntries = 0;  // fragments that pass the fill gate (after the strips took their rows)
    long long stripEntries = 0, stripBlocks = 0;     // binary16 strip chunks, or binary64 8 x 8 blocks (blocks64)
    long long stripBlocksOff = 0;                    // of stripBlocks: blocks of chunks that start off the grid of eight columns
    bool blocks64 = false;
    int dRows = 0, dCols = 0, nnzRowD = 0, frags = 0;  // what the extraction selected; fragments of the tile encoding
    std::vector<int> stripChunkBlocks, stripChunkEntries;  // per strip chunk, in layout order
};
struct HybridDevice {
    struct Impl;
    Impl *impl = nullptr;
    HybridDevice() = default;
    HybridDevice(const HybridDevice &) = delete;
    HybridDevice &operator=(const HybridDevice &) = delete;
    ~HybridDevice();
    // minVals: entries a fragment needs to pass the gate; want*: which forms the flags allow
    int analyse(mx_dtype dtype, int rows, int cols, int nnz, const int *rowPtr_dev, const int *col_dev, const void *val_dev, float tau_c,
                float tau_r, int minVals, bool wantGeneral, bool wantStrips, bool wantBlocks, HybridCounts *counts, hipStream_t s);
    // the same counts for an extraction that is there already: the arrays of `twin` are used where they are and
    // stay the twin's
    int adopt(const PartitionTwin &twin, int minVals, bool wantGeneral, bool wantStrips, bool wantBlocks, HybridCounts *counts, hipStream_t s);
    // stripRows_dev: marks of the rows the strips write (null when keepStrips is false or there are none).
    // keepGeneral: the fragments that pass the gate go to the general tile form -- tile_chunks and tile_layout
    // come first then, and the values of that layout are filled here.
    // keepBlocks (binary64, alone): the entries of the 8 x 8 blocks leave the CSR part and the rows of block chunks are
    // marked 2 -- block_chunks comes first then.
    int csr_part(bool keepStrips, bool keepGeneral, bool keepBlocks, int **rowPtr_dev, int **col_dev, void **val_dev, int *nnz,
                 char **stripRows_dev);
    // the binary64 block form: blocks per block row that has any and those block rows (ascending); then the layout
    // from the caller's steps (10 ints per step as for tile_layout)
    int block_chunks(std::vector<int> &blocks, std::vector<int> &blockRows);
    int block_layout(const std::vector<int> &stepDesc, const std::vector<int> &chunkBlock0, const std::vector<int> &waveDesc,
                     long long totalBlocks, DeviceTiles &T);
    // the general tile form: blocks per chunk that has any (chunk order); then the layout from the caller's steps --
    // stepDesc has 10 ints per step: the 8 of strip_layout with chunks numbered as in `blocks`, then the first block
    // of half 0 inside its chunk (a chunk of more blocks than a step holds takes several), then 0
    int tile_chunks(bool keepStrips, std::vector<int> &blocks);
    int tile_layout(bool keepStrips, const std::vector<int> &stepDesc, const std::vector<int> &chunkBlock0, const std::vector<int> &waveDesc,
                    long long totalBlocks, DeviceTiles &T);
    // stepDesc: 8 ints per step {chunk of half 0, chunk of half 1 (-1 none, -2 the first goes on), flags, blocks in half 0,
    // blocks in half 1, first value, first value and blocks in half 0 of the step four further on}; chunkBlock0: first block
    // of every chunk; T receives waveDesc, hdr, atox and tcVal
    int strip_layout(const std::vector<int> &stepDesc, const std::vector<int> &chunkBlock0, const std::vector<int> &waveDesc,
                     long long totalBlocks, DeviceTiles &T);
};

// `what`: 0 = slice kernel then combine kernel, 1 = slice kernel only, 2 = combine kernel only
// `strips` (optional): a tile layout in the dense binary16 form whose steps workgroups of the
// combine kernel's launch run as well (strips_can_ride says whether a layout may); the rows of
// those strips must be marked in the slice layout (rowInfo -2) so that the combine kernel leaves
// them alone.
// `ywide` (optional, all three launchers): an array of accumulators (binary32 for binary16
// plans), one per row.  The CSR launchers also store every sum they write to y there,
// unrounded; the tile launcher reads the old y of its rows from there instead of y, so that a
// row which gets sums from both parts is rounded to the value type once.
hipError_t launch_slices(mx_dtype dtype, const DeviceSlices &P, const void *x, void *y, int accumulate, hipStream_t s,
                         int what = 0, const DeviceTiles *strips = nullptr, void *ywide = nullptr);
// Raises the dynamic-LDS limit of the slice kernels on the current device (idempotent).  Every route that makes
// a DeviceSlices calls it before handing the layout out; launch_slices and launch_fused rely on that.
hipError_t prepare_slice_kernels(mx_dtype dtype);
// The one-launch form of the same product (P.fused).  `misplaced`: a word in host memory that the
// device can write (one per process); a workgroup that finds itself on another XCD than the layout
// assumes sets it, and the product of that launch cannot be trusted.
// `seq`: how many one-launch products of this layout were queued before this one (the kernel holds
// the claims of its logical workgroups against it).
hipError_t launch_fused(mx_dtype dtype, const DeviceSlices &P, const void *x, void *y, int accumulate, hipStream_t s,
                        void *ywide, unsigned *misplaced, unsigned seq);
// Whether the workgroups of a launch of `nWG` workgroups shaped like the one-launch form's take every
// logical workgroup (XCC_ID, blockIdx / 8) exactly once on the current device (asked once per device
// and grid size, by launching a probe that reads the XCC_ID register); *ok = 0 when not -- a device
// without eight XCDs, or a dispatcher that does not deal workgroups round-robin.
hipError_t fused_placement_ok(int nWG, int *ok);
bool strips_can_ride(mx_dtype dtype, const DeviceTiles &T, const void *x);
hipError_t launch_csr(mx_dtype dtype, const DeviceCsr &A, const void *x, void *y, int accumulate, hipStream_t s,
                      void *ywide = nullptr);
hipError_t launch_tiles(mx_dtype dtype, const DeviceTiles &T, const void *x, void *y, int accumulate, hipStream_t s,
                        const void *ywide = nullptr);
hipError_t launch_probe_f64(const double *A, const double *B, double *D, hipStream_t s);
hipError_t launch_probe_f16(const void *A, const void *B, float *D, hipStream_t s);

}  // namespace mx

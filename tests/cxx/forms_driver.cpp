// How a plan looks for the forms of its CSR part that are made on the device (mxp::try_forms), with the two makers
// replaced by what the check says.  No GPU call.  Run with the name of one check; exit status 0 means it holds.
#include <algorithm>
#include <cstdio>
#include <cstdlib>
#include <map>
#include <string>
#include <vector>

#include "mx_plan_parts.h"

#define CHECK(x)                                                     \
    do {                                                             \
        if (!(x)) {                                                  \
            std::printf("line %d: %s does not hold\n", __LINE__, #x); \
            std::exit(1);                                            \
        }                                                            \
    } while (0)

namespace {
int offsets_rc = MX_OK, windows_rc = MX_OK, offsets_asked = 0, windows_asked = 0;
bool offsets_suit = false, windows_suit = false;
}  // namespace

namespace mx {
int build_offsets_device(mx_dtype, int, int, int, const int *, const int *, const void *, DeviceOffsets &D, hipStream_t)
{
    ++offsets_asked;
    D = DeviceOffsets();
    if (offsets_suit) D.nChunks = 5;
    return offsets_rc;
}
int build_windows_device(mx_dtype, int, int, int, const int *, const int *, const void *, DeviceWindows &D, hipStream_t)
{
    ++windows_asked;
    D = DeviceWindows();
    if (windows_suit) D.nChunks = 7;
    return windows_rc;
}
hipError_t launch_offsets(mx_dtype, const DeviceOffsets &, const void *, void *, hipStream_t) { return hipErrorUnknown; }
hipError_t launch_windows(mx_dtype, const DeviceWindows &, const void *, void *, hipStream_t) { return hipErrorUnknown; }
}  // namespace mx

// No memory for a form is a reason to go on without it (the forms behind it need less beside the matrix), any other
// failure is the plan's.
static void no_memory()
{
    const struct {
        int orc, wrc;
        bool osuit, wsuit;
        int rc, variant;
    } cases[] = {
        {MX_OK, MX_OK, true, true, MX_OK, 3},
        {MX_OK, MX_OK, false, true, MX_OK, 4},
        {MX_OK, MX_OK, false, false, MX_OK, 0},
        {MX_ERR_ALLOC, MX_OK, true, true, MX_OK, 4},
        {MX_ERR_ALLOC, MX_OK, true, false, MX_OK, 0},
        {MX_OK, MX_ERR_ALLOC, false, true, MX_OK, 0},
        {MX_ERR_ALLOC, MX_ERR_ALLOC, true, true, MX_OK, 0},
        {MX_ERR_DEVICE, MX_OK, true, true, MX_ERR_DEVICE, 0},
        {MX_OK, MX_ERR_DEVICE, false, true, MX_ERR_DEVICE, 0},
    };
    for (const auto &c : cases) {
        offsets_rc = c.orc, windows_rc = c.wrc, offsets_suit = c.osuit, windows_suit = c.wsuit;
        mx_plan plan;
        plan.rows = plan.cols = 100000;
        bool took = false;
        CHECK(mxp::try_forms(&plan, 1000000, nullptr, nullptr, nullptr, MX_PLAN_DEFAULT, &took) == c.rc);
        CHECK(plan.csr_variant == c.variant && took == (c.rc == MX_OK && c.variant != 0));
        if (c.rc == MX_OK) CHECK((plan.offsets.nChunks > 0) == (c.variant == 3) && (plan.windows.nChunks > 0) == (c.variant == 4));
    }
}

// The window form where it was measured to be faster than slices or row tiles, and not where it was slower.  `lines`: of x, per gather of
// 64 entries, as such a band has them.
static void window_rule()
{
    const struct {
        bool f64;
        int rows, nnz;
        double stored;  // MB
        double lines;
        bool pays;
    } cases[] = {
        // (faster)
        {true, 66000, 2640000, 26.5, 55, true},     {true, 33000, 3300000, 32.5, 55, true},     {true, 130000, 39000000, 385.9, 60, true},
        {true, 600000, 9600000, 99.7, 50, true},    {true, 600000, 4788000, 50.0, 50, true},    {true, 260000, 10400000, 105.5, 60, true},
        {false, 250007, 10000280, 42.0, 55, true},  {false, 130000, 780000, 4.3, 25, true},     {false, 66000, 6600000, 26.2, 60, true},
        {false, 600000, 23844517, 115.4, 50, true}, {false, 1500000, 23940000, 97.4, 45, true}, {false, 400000, 3188000, 13.0, 45, true},
        // (slower)
        {true, 33000, 9228706, 136.4, 60, false},   {true, 66000, 18793119, 193.7, 60, false},  {true, 600000, 23840358, 314.4, 58, false},
        {true, 260000, 1549859, 21.1, 36, false},   {true, 1500000, 8943723, 122.5, 40, false}, {true, 400000, 2376000, 33.0, 28, false},
        {true, 260000, 25561141, 383.1, 60, false}, {false, 33000, 8628000, 51.6, 60, false},   {false, 3200000, 28679476, 156.0, 40, false},
        {false, 3200000, 22330908, 104.0, 40, false}, {false, 130000, 37423087, 222.9, 60, false},
    };
    for (const auto &c : cases) {
        const int nWG = ((c.rows + 63) / 64 + mx::kWindowWaves - 1) / mx::kWindowWaves;
        const double other = mx::other_forms_us(c.f64 ? MX_F64 : MX_F16, c.rows, c.rows, c.nnz, c.lines), touched = c.stored * 1e6 + 2.0 * c.rows * (c.f64 ? 8 : 2);
        const bool pays = mx::window_form_pays(c.f64, c.nnz, c.stored * 1e6, touched, nWG, 256, other);
        if (pays != c.pays)
            std::printf("binary%d, %d rows, %d entries, %.1f MB: %.1f us, otherwise %.1f\n", c.f64 ? 64 : 16, c.rows, c.nnz, c.stored,
                        mx::window_estimate(c.f64, c.stored * 1e6, touched, nWG, 256), other);
        CHECK(pays == c.pays);
    }
}

// Plain or streaming loads, by what the form itself was measured at.
static void keep_rule()
{
    mx_plan plan;
    plan.dtype = MX_F16;
    plan.rows = plan.cols = 1000000;
    const struct {
        int variant;
        double mb;
        bool keep;
    } cases[] = {{3, 100, true}, {3, 130, true}, {3, 140, false}, {4, 100, true}, {4, 130, true}, {4, 140, false}};
    for (const auto &c : cases) {
        plan.csr_variant = c.variant;
        const double rest = c.mb * 1e6 - 4e6;  // (x and y)
        plan.offsets.units = (int)(rest / (64 * 16)), plan.offsets.unitBytes = 16;
        plan.windows.units = (int)(rest / 1024), plan.windows.unitBytes = 1024;
        mxp::decide_keep(&plan, MX_PLAN_DEFAULT);
        CHECK((c.variant == 3 ? plan.offsets.keep : plan.windows.keep) == c.keep);
    }
}

// Waves that share a chunk of the offset form: one where its list is one round.
static void offset_waves()
{
    CHECK(mx::offsets_waves(true, false, 11719, 11719) == 1 && mx::offsets_waves(true, false, 8 * 11719, 11719) == 1);
    CHECK(mx::offsets_waves(true, false, 9 * 11719, 11719) == 4 && mx::offsets_waves(true, true, 12 * 11719, 11719) == 2);
    CHECK(mx::offsets_waves(true, true, 8 * 11719, 11719) == 1 && mx::offsets_waves(true, true, 12 * 300, 300) == 4);
    CHECK(mx::offsets_waves(false, false, 8 * 5860, 5860) == 1 && mx::offsets_waves(false, true, 28 * 5860, 5860) == 4);
    CHECK(mx::offsets_waves(true, false, 8ll << 28, 1 << 28) == 1);
    CHECK(mx::offsets_waves(false, false, 8 * 470, 470) == 4 && mx::offsets_waves(true, true, 8 * 235, 235) == 4);
    CHECK(mx::offsets_waves(false, false, 4 * 470, 470) == 1 && mx::offsets_waves(true, false, 8 * 1400, 1400) == 1);
}

// Long lists on small matrices, where row tiles were measured to be the faster ones.
static void offset_lists()
{
    CHECK(!mx::offsets_lists_pay(true, false, 60, 65100) && !mx::offsets_lists_pay(true, false, 48, 480000));
    CHECK(mx::offsets_lists_pay(true, false, 27, 27000) && mx::offsets_lists_pay(true, false, 60, 1200000));
    CHECK(mx::offsets_lists_pay(true, true, 60, 299100) && mx::offsets_lists_pay(true, false, 48, 960000));
    CHECK(!mx::offsets_lists_pay(false, false, 60, 600000) && !mx::offsets_lists_pay(false, true, 60, 299100));
    CHECK(mx::offsets_lists_pay(false, false, 48, 240000) && mx::offsets_lists_pay(false, true, 60, 1800000));
}

// What a plan says of the workgroups of its CSR kernel is what the launch has.
static void csr_blocks()
{
    mx_plan plan;
    mx_plan_info info;
    plan.rows = plan.cols = 1500000;
    plan.csr_variant = 3;
    plan.offsets.nChunks = 11719;
    const struct {
        int perChunk, nDict, blocks;
    } cases[] = {{3, 0, 2930}, {27, 0, 11719}, {28, 2, 5860}};
    for (const auto &c : cases) {
        plan.offsets.nOffs = (long long)c.perChunk * plan.offsets.nChunks;
        plan.offsets.nDict = c.nDict;
        CHECK(mx_plan_get_info(&plan, &info) == MX_OK && info.csr_blocks == c.blocks);
    }
    plan.csr_variant = 4;
    plan.windows.nWG = 489, plan.windows.nApart = 11;
    CHECK(mx_plan_get_info(&plan, &info) == MX_OK && info.csr_blocks == 500);
}

// The entries that one thread of a kernel looks at: all below n and n at the end, also where n is close to what an int
// holds (2^31 - 513 entries are accepted): by the threads of a grid of 1024 workgroups, of a workgroup, of four entries on their way for each of its
// threads, by tiles of 8192.
static void strides()
{
    const int n = 2147483647 - 512;
    for (const int stride : {1024 * 256, 1024, 4 * 256, 8192})
        for (const int first : {n - 3000000, n - 3000000 + stride - 1, n - 1, n - stride - 1, n - stride, n - stride + 1}) {
            int p = first, steps = 0;
            for (; p < n; p = mx::next_of(p, n, stride)) {
                CHECK(p >= 0);
                CHECK(++steps <= 3000000 / stride + 2);
            }
            CHECK(p == n && steps == (n - 1 - first) / stride + 1);
        }
    // the first of a thread, in a stretch that begins among the last places
    for (const int p0 : {n - 5000, n - 1024, n - 1023, n - 1, n})
        for (const int thread : {0, 1, 255, 1023, 1024}) CHECK(mx::next_of(p0, n, thread) == (thread < n - p0 ? p0 + thread : n));
    CHECK(mx::next_of(5, 3, 2) == 3 && mx::next_of(0, 1, 262144) == 1);
    // ... and matrices whose last chunk would not be numbered in an int do not take the forms
    CHECK(mx::forms_can_number(n, n, n) && !mx::forms_can_number(n + 1, 5, 5) && !mx::forms_can_number(5, n + 1, 5) && !mx::forms_can_number(5, 5, n + 1));
}

// Every column falls into one of the window form's buckets, of whole vectors of x.
static void window_buckets()
{
    for (const int epv : {2, 8})
        for (const int cols : {64, 2047, 2048, 2049, 16384, 16385, 30011, 1000003, 2147483647 - 2048, 2147483647 - 2047, 2147483647 - 512}) {
            const int size = mx::window_bucket(cols, epv);
            CHECK(size >= epv && size % epv == 0 && (cols - 1) / size < mx::kWindowBuckets);
            CHECK(size == epv || (long long)(size - epv) * mx::kWindowBuckets < cols);  // (no larger than it has to be)
        }
}

// What the host can tell of a matrix before it is sent up for the forms: never "no" to one that a form takes.
static void host_look()
{
    struct Matrix {
        int rows, cols;
        std::vector<int> ptr{0}, col;
        Matrix(int r, int c) : rows(r), cols(c) {}
        void end_row() { ptr.push_back((int)col.size()); }
        bool may(mx_dtype t) const { return mxp::forms_may_suit(t, rows, cols, ptr.data(), col.data()); }
    };
    unsigned seed = 1;
    auto random = [&](int n) { return (int)((seed = seed * 1664525u + 1013904223u) >> 8) % n; };
    auto uniform = [&](int rows, int cols, int per) {
        Matrix A(rows, cols);
        for (int r = 0; r < rows; ++r, A.end_row())
            for (int k = 0; k < per; ++k) A.col.push_back(random(cols));
        return A;
    };
    auto band = [&](int rows, int per, int half) {
        Matrix A(rows, rows);
        for (int r = 0; r < rows; ++r, A.end_row())
            for (int k = 0; k < per; ++k) A.col.push_back(std::min(std::max(r + random(2 * half + 1) - half, 0), rows - 1));
        return A;
    };
    auto diagonals = [&](int rows, int n) {
        Matrix A(rows, rows);
        for (int r = 0; r < rows; ++r, A.end_row())
            for (int k = 0; k < n; ++k)
                if (r + k - n / 2 >= 0 && r + k - n / 2 < rows) A.col.push_back(r + k - n / 2);
        return A;
    };
    for (const mx_dtype t : {MX_F64, MX_F16}) {
        CHECK(diagonals(5000, 64).may(t) && !diagonals(5000, 65).may(t) && diagonals(1024, 1).may(t) && !diagonals(1023, 1).may(t));
        CHECK(band(40000, 20, 500).may(t) && band(40000, 20, 3000).may(t) && !band(30000, 20, 500).may(t));
        CHECK(!uniform(4096, 4096, 16).may(t) && !uniform(65536, 65536, 16).may(t) && !uniform(40000, 300000, 30).may(t) && !uniform(2000, 50, 80).may(t));
        Matrix far = band(40000, 20, 500);  // a few rows of another kind are no reason
        for (int p = 0; p < 40000; p += 997) far.col[p] = random(40000);
        CHECK(far.may(t));
        Matrix longRow = band(40000, 20, 500);
        for (int k = 0; k < 1025; ++k) longRow.col.push_back(k);
        longRow.ptr.back() = (int)longRow.col.size();
        CHECK(!longRow.may(t));
        Matrix empty(50000, 50000);
        for (int r = 0; r < 50000; ++r) empty.end_row();
        CHECK(!empty.may(t));
    }
}

int main(int argc, char **argv)
{
    const std::map<std::string, void (*)()> checks = {{"no_memory", no_memory}, {"window_rule", window_rule}, {"keep_rule", keep_rule}, {"offset_waves", offset_waves}, {"offset_lists", offset_lists}, {"csr_blocks", csr_blocks}, {"strides", strides}, {"window_buckets", window_buckets}, {"host_look", host_look}};
    const auto it = checks.find(argc > 1 ? argv[1] : "");
    if (it == checks.end()) return 2;
    it->second();
    return 0;
}

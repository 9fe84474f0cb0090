// Where the CSR part of a plan is laid out when the matrix is in host memory (mxp::setup_csr_part), on a device that exists only
// here: the HIP functions on that path are defined below and count bytes, and the layouts that the device makes are replaced by what the
// check says.  Run with the name of one check; exit status 0 means it holds.
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <map>
#include <new>
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
struct Device {
    size_t total = (size_t)4 << 30, used = 0;
    std::map<void *, size_t> blocks;
    hipError_t last = hipSuccess;
} device;
int slices_rc = MX_OK, rows_rc = MX_OK, slices_asked = 0, rows_asked = 0;
bool slices_throw = false;
}  // namespace

extern "C" {
hipError_t hipGetDevice(int *d) { return *d = 0, hipSuccess; }
hipError_t hipGetDeviceCount(int *n) { return *n = 1, hipSuccess; }
hipError_t hipDeviceGetAttribute(int *v, hipDeviceAttribute_t, int) { return *v = 256, hipSuccess; }
hipError_t hipDeviceSynchronize() { return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipStreamIsCapturing(hipStream_t, hipStreamCaptureStatus *s) { return *s = hipStreamCaptureStatusNone, hipSuccess; }
hipError_t hipMemGetInfo(size_t *f, size_t *t) { return *f = device.total - device.used, *t = device.total, hipSuccess; }
hipError_t hipMalloc(void **p, size_t n)
{
    if (device.used + n > device.total) return device.last = hipErrorOutOfMemory;
    *p = std::malloc(n);
    CHECK(*p);
    device.blocks[*p] = n;
    device.used += n;
    return hipSuccess;
}
hipError_t hipFree(void *p)
{
    const auto it = device.blocks.find(p);
    CHECK(it != device.blocks.end());
    device.used -= it->second;
    device.blocks.erase(it);
    std::free(p);
    return hipSuccess;
}
hipError_t hipMemcpy(void *to, const void *from, size_t n, hipMemcpyKind) { return std::memcpy(to, from, n), hipSuccess; }
hipError_t hipMemset(void *to, int v, size_t n) { return std::memset(to, v, n), hipSuccess; }
const char *hipGetErrorString(hipError_t) { return ""; }
hipError_t hipGetLastError()
{
    const hipError_t e = device.last;
    device.last = hipSuccess;
    return e;
}
}

namespace mx {
int build_offsets_device(mx_dtype, int, int, int, const int *, const int *, const void *, DeviceOffsets &D, hipStream_t) { return D = DeviceOffsets(), MX_OK; }
int build_windows_device(mx_dtype, int, int, int, const int *, const int *, const void *, DeviceWindows &D, hipStream_t) { return D = DeviceWindows(), MX_OK; }
hipError_t launch_offsets(mx_dtype, const DeviceOffsets &, const void *, void *, hipStream_t) { return hipErrorUnknown; }
hipError_t launch_windows(mx_dtype, const DeviceWindows &, const void *, void *, hipStream_t) { return hipErrorUnknown; }
hipError_t fused_placement_ok(int, int *ok) { return *ok = 0, hipSuccess; }
int lines_per_gather_device(mx_dtype, int, const int *, hipStream_t, double *out) { return *out = 8.0, MX_OK; }
int build_slices_device(mx_dtype, int rows, int, int, const int *, const int *, const void *, int, int, const char *, DeviceSlices &D, hipStream_t,
                        std::vector<int> *, std::vector<int> *, int)
{
    ++slices_asked;
    if (slices_throw) throw std::bad_alloc();
    D = DeviceSlices();
    D.vrows = 4 * rows;
    if (dev_malloc((void **)&D.ecol, 1000) != hipSuccess) return MX_ERR_ALLOC;
    return slices_rc;
}
int upload_csr_device(mx_dtype, int rows, int cols, int nnz, const int *, const int *, const void *, const std::vector<int> &, bool, DeviceCsr &A, hipStream_t)
{
    ++rows_asked;
    A = DeviceCsr();
    A.rows = rows, A.cols = cols, A.nnz = nnz;
    if (dev_malloc((void **)&A.rowPtr, 1000) != hipSuccess) return MX_ERR_ALLOC;
    return rows_rc;
}
}  // namespace mx

namespace {
// 64 columns side by side in every row (row tiles are the faster form by far), distinct values, a million entries and more
struct Band {
    int rows = 20000, cols = 20064;
    std::vector<int> ptr, col;
    std::vector<double> val;
    Band()
    {
        ptr.push_back(0);
        for (int r = 0; r < rows; ++r) {
            for (int k = 0; k < 64; ++k) col.push_back(r + k), val.push_back(0.5 + 1e-6 * (double)col.size());
            ptr.push_back((int)col.size());
        }
    }
    size_t raw() const { return (ptr.size() + col.size()) * 4 + val.size() * 8; }
};
const Band &band()
{
    static const Band b;
    return b;
}
// A plan's CSR part from the matrix; the device's layouts that were asked for on the way.
int made(mx_plan &plan, int flags)
{
    const Band &b = band();
    plan.dtype = MX_F64;
    plan.rows = b.rows, plan.cols = b.cols, plan.nnz = (int)b.col.size();
    slices_asked = rows_asked = 0;
    mx::MemScope scope(nullptr);
    return mxp::setup_csr_part(&plan, b.ptr.data(), b.col.data(), b.val.data(), flags);
}
void dropped(mx_plan &plan)
{
    mxp::free_csr(plan.csr);
    mxp::free_slices(plan.slices);
    mx::release_idle_memory();
    CHECK(device.used == 0);
}
}  // namespace

// Too many places for the slices is the slices' matter: the part has its row tiles all the same.
static void refused()
{
    {
        mx_plan plan;
        slices_rc = rows_rc = MX_OK;
        CHECK(made(plan, MX_PLAN_DEFAULT) == MX_OK && slices_asked == 1 && rows_asked == 1 && plan.csr_variant == 0);
        dropped(plan);
    }
    mx_plan plan;
    slices_rc = MX_ERR_ARG;
    CHECK(made(plan, MX_PLAN_DEFAULT) == MX_OK);
    CHECK(slices_asked == 1 && rows_asked == 0);  // (the host's route has estimated first)
    CHECK(plan.csr_variant == 0 && plan.csr.rows == band().rows && plan.csr.nBlocks > 0 && !plan.slices.ecol);
    dropped(plan);
    // whoever asks for slices is refused
    CHECK(made(plan, MX_PLAN_CSR_SLICES) == MX_ERR_ARG);
    dropped(plan);
    slices_rc = MX_ERR_DEVICE;  // (any other failure is the plan's)
    CHECK(made(plan, MX_PLAN_DEFAULT) == MX_ERR_DEVICE && slices_asked == 1);
    dropped(plan);
}

// A device without room for the matrix beside the plan, or that runs out while it lays the plan out: the part has its row tiles all the same.
static void memory()
{
    const Band &b = band();
    slices_rc = rows_rc = MX_OK;
    for (const int flags : {MX_PLAN_DEFAULT, MX_PLAN_CSR_ROWS}) {
        const size_t tiles = b.ptr.size() * 4 + (b.col.size() + mx::kCsrPad) * (sizeof(double) + 2) + 1000000;  // (16-bit columns)
        CHECK(tiles < b.raw());
        device.total = tiles;
        {
            mx_plan plan;
            CHECK(made(plan, flags) == MX_OK && slices_asked + rows_asked == 0 && plan.csr_variant == 0 && plan.csr.nBlocks > 0);
            dropped(plan);
        }
        device.total = b.raw() / 2;  // (nor for the tiles)
        {
            mx_plan plan;
            CHECK(made(plan, flags) != MX_OK);
            dropped(plan);
        }
        device.total = (size_t)4 << 30;
        rows_rc = MX_ERR_ALLOC;
        mx_plan plan;
        CHECK(made(plan, flags) == MX_OK && rows_asked == 1 && plan.csr_variant == 0 && plan.csr.nBlocks > 0);
        dropped(plan);
        rows_rc = MX_OK;
    }
    // host memory that runs out meanwhile leaves nothing behind on the device
    slices_throw = true;
    mx_plan plan;
    bool thrown = false;
    try {
        (void)made(plan, MX_PLAN_DEFAULT);
    } catch (const std::bad_alloc &) {
        thrown = true;
    }
    slices_throw = false;
    CHECK(thrown);
    dropped(plan);
}

// What the device's kernels cannot number does not go up.
static void sizes()
{
    const int n = 2147483647 - 512;
    CHECK(mxp::part_goes_up(5, 5, 1 << 20) && !mxp::part_goes_up(5, 5, (1 << 20) - 1) && mxp::part_goes_up(n, n, n));
    CHECK(!mxp::part_goes_up(n + 1, 5, 1 << 20) && !mxp::part_goes_up(5, n + 1, 1 << 20) && !mxp::part_goes_up(5, 5, n + 1));
}

int main(int argc, char **argv)
{
    const std::map<std::string, void (*)()> checks = {{"refused", refused}, {"memory", memory}, {"sizes", sizes}};
    const auto it = checks.find(argc > 1 ? argv[1] : "");
    if (it == checks.end()) return 2;
    it->second();
    return 0;
}

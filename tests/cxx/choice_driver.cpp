// Where matxtract_preprocess makes the extraction, with a device that exists only here: the two calls by which it reaches one
// are answered below.  Exit status 0 means all checks hold.
#include <cstdio>
#include <cstdlib>
#include <vector>

#include "MatXtract.h"

static int asked = 0, answer = MX_ERR_ALLOC;
extern "C" int mx_device_count(void) { return 1; }
extern "C" int mx_partition_create_device(const mx_csr *, float, float, mx_partition **out)
{
    ++asked;
    *out = nullptr;
    return answer;
}

#define CHECK(x)                                                     \
    do {                                                             \
        if (!(x)) {                                                  \
            std::printf("line %d: %s does not hold\n", __LINE__, #x); \
            std::exit(1);                                            \
        }                                                            \
    } while (0)

int main()
{
    const int rows = 40000, per = 8;  // (320000 entries)
    std::vector<indT> ptr(rows + 1), col((size_t)rows * per);
    std::vector<valT> val((size_t)rows * per, valT{});
    for (int r = 0; r < rows; ++r) {
        ptr[r + 1] = (r + 1) * per;
        for (int k = 0; k < per; ++k) col[(size_t)r * per + k] = (indT)((r * 7 + k * k * 11) % rows);
    }
    auto make = [&](int r, float c, int on) { return matxtract_preprocess(val.data(), ptr.data(), col.data(), r, rows, r * per, c, c, on); };
    for (const int code : {MX_ERR_ALLOC, MX_ERR_DEVICE}) {
        answer = code;
        asked = 0;
        mx_partition *p = make(rows, 0.5f, -1), *q = make(rows, 0.5f, 0);
        CHECK(p && q && asked == 1 && mx_partition_hash(p) == mx_partition_hash(q));
        mx_partition_destroy(p);
        mx_partition_destroy(q);
        CHECK(!make(rows, 0.5f, 1) && asked == 2);  // (whoever asks for the device is told)
    }
    answer = MX_ERR_ARG;
    asked = 0;
    CHECK(!make(rows, 0.5f, -1) && asked == 1);
    mx_partition *p = make(1000, 0.5f, -1), *q = make(rows, 0.0f, -1);  // small, or nothing to extract
    CHECK(p && q && asked == 1);
    mx_partition_destroy(p);
    mx_partition_destroy(q);
    std::printf("ok\n");
    return 0;
}

// Host check of the job tables and keyed tables (mpsq_buffers.h) over a stand-in for the
// HIP runtime whose "device" is host memory: equal tables are not uploaded
// again, changed ones are, and after a fill that was cut short by a failed
// allocation the device still ends with the tables of the next run.  Prints
// "ok" or the first failure.
#include <cstdio>
#include <cstdlib>
#include <cstring>

enum hipError_t { hipSuccess = 0, hipErrorOutOfMemory = 2 };
enum hipMemcpyKind { hipMemcpyHostToDevice };
typedef struct Stream *hipStream_t;
typedef struct Event *hipEvent_t;
constexpr unsigned hipHostMallocDefault = 0, hipEventDisableTiming = 2;
constexpr int MPSQ_ERR_DEVICE = 5;
static int fail_host = -1, fail_dev = -1, copies = 0;  // allocations left before one fails; copies made
static hipError_t get(void **p, size_t n, int &left)
{
    if (left >= 0 && left-- == 0) return hipErrorOutOfMemory;
    *p = std::calloc(1, n);
    return hipSuccess;
}
static hipError_t hipHostMalloc(void **p, size_t n, unsigned) { return get(p, n, fail_host); }
static hipError_t hipMalloc(void **p, size_t n) { return get(p, n, fail_dev); }
static hipError_t hipFree(void *p) { std::free(p); return hipSuccess; }
static hipError_t hipHostFree(void *p) { std::free(p); return hipSuccess; }
static hipError_t hipEventCreateWithFlags(hipEvent_t *e, unsigned) { *e = reinterpret_cast<hipEvent_t>(1); return hipSuccess; }
static hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
static hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
static hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
static hipError_t hipMemcpyAsync(void *d, const void *s, size_t n, hipMemcpyKind, hipStream_t)
{
    ++copies;
    std::memcpy(d, s, n);
    return hipSuccess;
}

#include "mpsq_buffers.h"

using namespace mpsq;

static std::vector<int> table(int n, int v) { return std::vector<int>((size_t)n, v); }

// one run's tables; false if the fill threw
static bool fill(Arena &A, const std::vector<std::vector<int>> &ts, hipStream_t st)
{
    try {
        A.begin();
        for (const auto &t : ts) A.put(t);
        A.upload(st);
        return true;
    } catch (const Err &) {
        return false;
    }
}

static bool same(const Arena &A, const std::vector<std::vector<int>> &ts)
{
    size_t off = 0;
    for (const auto &t : ts) {
        off = (off + 255) & ~(size_t)255;
        if (std::memcmp(A.dev<int>(off), t.data(), 4 * t.size()) != 0) return false;
        off += 4 * t.size();
    }
    return true;
}

#define CHECK(x)                                                                                                      \
    if (!(x)) {                                                                                                       \
        std::printf("FAIL line %d: %s\n", __LINE__, #x);                                                              \
        return 1;                                                                                                     \
    }

int main()
{
    hipStream_t s1 = reinterpret_cast<hipStream_t>(1), s2 = reinterpret_cast<hipStream_t>(2);
    const std::vector<std::vector<int>> a{table(100, 1), table(50, 2)}, b{table(100, 1), table(50, 3)},
        c{table(100, 1)}, big{table(100, 7), table(50, 8), table(1 << 20, 9)};
    {
        Arena A;
        CHECK(fill(A, a, s1) && copies == 1 && same(A, a));
        CHECK(fill(A, a, s1) && copies == 1);                 // equal: not sent again
        CHECK(fill(A, b, s1) && copies == 2 && same(A, b));
        CHECK(fill(A, c, s1) && copies == 2 && same(A, c));   // a part of what is there
        CHECK(fill(A, b, s1) && copies == 2 && same(A, b));
        CHECK(fill(A, b, s2) && copies == 3 && same(A, b));   // another stream
        CHECK(fill(A, big, s2) && copies == 4 && same(A, big));
    }
    {
        // the fill of other tables fails when they outgrow the host memory
        Arena A;
        CHECK(fill(A, a, s1) && same(A, a));
        fail_host = 0;
        CHECK(!fill(A, big, s1));
        fail_host = -1;
        const std::vector<std::vector<int>> part{big[0], big[1]};
        CHECK(fill(A, part, s1) && same(A, part));
        CHECK(fill(A, a, s1) && same(A, a));
    }
    {
        // the upload fails when the device memory cannot grow
        Arena A;
        CHECK(fill(A, a, s1) && same(A, a));
        fail_dev = 0;
        CHECK(!fill(A, big, s1));
        fail_dev = -1;
        CHECK(fill(A, big, s1) && same(A, big));
        CHECK(fill(A, a, s1) && same(A, a));
    }
    {
        // a table whose allocation failed is made anew, not taken for the old one
        KeyedTable<int> K;
        auto get = [&](int v, size_t n) -> const int * {
            try {
                return K.get({v, 0, 0}, n, s1, [&](int *h) { std::fill(h, h + n, v); });
            } catch (const Err &) {
                return nullptr;
            }
        };
        const int *p = get(3, 10);
        const int n0 = copies;
        CHECK(p && p[0] == 3 && p[9] == 3);
        CHECK(get(3, 10) == p && copies == n0);
        fail_dev = 0;
        CHECK(!get(4, 1000));
        fail_dev = -1;
        p = get(3, 10);
        CHECK(p && p[0] == 3 && p[9] == 3);
        p = get(4, 1000);
        CHECK(p && p[999] == 4);
    }
    std::printf("ok\n");
    return 0;
}

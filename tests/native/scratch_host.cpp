// The scratch of prims.hip on a stand-in for the HIP runtime: device memory is
// a byte count with a limit, launches do nothing, and a failed call's error
// stays with the thread until hipGetLastError reads it.
//   scratch_host CASE     (exit status 0: the case holds)
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <map>
#include <string>

#include "prims.hpp"

namespace fake {
size_t limit = (size_t)1 << 40, used = 0, most = 0;
std::map<void *, size_t> live;
thread_local hipError_t last = hipSuccess;
uintptr_t next = 4096;
}  // namespace fake

extern "C" {
hipError_t hipMalloc(void **p, size_t n)
{
    if (fake::used + n > fake::limit) return fake::last = hipErrorOutOfMemory;
    *p = (void *)fake::next;
    fake::next += (n + 8191) & ~(size_t)4095;
    fake::live[*p] = n;
    fake::used += n;
    if (fake::used > fake::most) fake::most = fake::used;
    return hipSuccess;
}
hipError_t hipFree(void *p)
{
    if (!fake::live.count(p)) std::abort();
    fake::used -= fake::live[p];
    fake::live.erase(p);
    return hipSuccess;
}
hipError_t hipGetDevice(int *d) { return *d = 0, hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipGetLastError() { hipError_t e = fake::last; fake::last = hipSuccess; return e; }
const char *hipGetErrorString(hipError_t) { return "error"; }
hipError_t hipMemcpyAsync(void *, const void *, size_t, hipMemcpyKind, hipStream_t) { return hipSuccess; }
hipError_t hipMemsetAsync(void *, int, size_t, hipStream_t) { return hipSuccess; }
hipError_t hipLaunchKernel(const void *, dim3, dim3, void **, size_t, hipStream_t) { return hipSuccess; }
hipError_t __hipPushCallConfiguration(dim3, dim3, size_t, hipStream_t) { return hipSuccess; }
hipError_t __hipPopCallConfiguration(dim3 *, dim3 *, size_t *, hipStream_t *) { return hipSuccess; }
void **__hipRegisterFatBinary(const void *) { return nullptr; }
void __hipRegisterFunction(void **, const void *, char *, const char *, unsigned, void *, void *, void *, void *, int *) {}
void __hipUnregisterFatBinary(void **) {}
}

using namespace abhsf;

#define CHECK(c)                                                     \
    do {                                                             \
        if (!(c)) {                                                  \
            std::printf("line %d: %s does not hold\n", __LINE__, #c); \
            return 1;                                                \
        }                                                            \
    } while (0)

constexpr size_t MiB = (size_t)1 << 20;

// One operation that used pieces of these sizes (MiB).
static void operation(std::initializer_list<size_t> sizes)
{
    Arena a(nullptr);
    for (size_t n : sizes) a.take_bytes(n * MiB);
}

// An allocation that succeeds after the kept scratch is freed leaves no error
// behind for the next launch check; nor does one that fails for good.
static int retry()
{
    operation({64, 32});
    fake::limit = 120 * MiB;
    DevBuf b(100 * MiB);
    CHECK(b.get() != nullptr);
    CHECK(hipGetLastError() == hipSuccess);
    bool thrown = false;
    try {
        DevBuf c(100 * MiB);
    } catch (const Error &e) {
        thrown = e.code == ABHSF_ERR_ALLOC;
    }
    CHECK(thrown);
    CHECK(hipGetLastError() == hipSuccess);
    return 0;
}

// Kept buffers that an open operation has not taken are freed when memory runs
// out; one that it needs is taken, and one that it did not need is gone after.
static int idle()
{
    operation({300, 200});
    CHECK(fake::used == 500 * MiB);
    {
        Arena a(nullptr);
        a.take_bytes(200 * MiB);
        CHECK(fake::used == 500 * MiB);  // the kept one
        fake::limit = 600 * MiB;
        DevBuf b(350 * MiB);
        CHECK(fake::used == 550 * MiB);
    }
    CHECK(fake::used == 200 * MiB);
    operation({90, 50});
    CHECK(fake::used == 140 * MiB);
    fake::limit = (size_t)1 << 40;
    operation({600, 600});  // above the bound: one of them
    CHECK(fake::used == 600 * MiB);
    return 0;
}

// What the sort took is not held for the rest of its operation: later pieces
// take its place, and an allocation that needs the memory gets it.
static int sorted()
{
    constexpr uint64_t n = (uint64_t)16 << 20;
    Arena a(nullptr);
    uint64_t *keys = a.take<uint64_t>(n);
    uint32_t *vals = a.take<uint32_t>(n);
    const size_t before = fake::used;
    radix_sort_pairs(keys, vals, n, 24, nullptr, a);
    const size_t after = fake::used;
    CHECK(after >= before + 12 * n);
    a.take<uint64_t>(n);
    CHECK(fake::used == after);
    fake::limit = after;
    DevBuf b(4 * n);  // the sort's second values
    CHECK(fake::used <= after);
    return 0;
}

// A piece does not hold a kept buffer much larger than itself.
static int fitting()
{
    operation({200});
    fake::limit = 250 * MiB;
    Arena a(nullptr);
    a.take_bytes(100 * MiB);
    DevBuf b(120 * MiB);
    CHECK(fake::used == 220 * MiB);
    return 0;
}

// The call that gives the memory back says how much it was; an operation that
// runs goes on.
static int trim()
{
    operation({64, 32});
    Arena a(nullptr);
    void *p = a.take_bytes(32 * MiB);
    CHECK(scratch_trim() == 64 * MiB);
    CHECK(fake::used == 32 * MiB && fake::live.count(p));
    {
        const Arena::Scope scope(a);
        a.take_bytes(40 * MiB);
    }
    CHECK(scratch_trim() == 40 * MiB);
    CHECK(scratch_trim() == 0);
    return 0;
}

int main(int argc, char **argv)
{
    const std::string c = argc > 1 ? argv[1] : "";
    if (c == "retry") return retry();
    if (c == "idle") return idle();
    if (c == "sorted") return sorted();
    if (c == "fitting") return fitting();
    if (c == "trim") return trim();
    return 2;
}

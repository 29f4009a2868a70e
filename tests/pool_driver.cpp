// The device memory pool of common.cpp over a HIP runtime made of counters: what
// it hands on, when it waits, what it keeps and what it gives back.
#include <cstdio>
#include <cstdlib>
#include <map>

#include "ra_internal.hpp"

namespace {
std::map<void*, size_t> allocated;  // live allocations
size_t total = 0, limit = size_t(64) << 30, last_size = 0;
int waits = 0, frees = 0;
bool capturing = false;
hipError_t last_error = hipSuccess;
uintptr_t next_address = 4096;

hipError_t fail_with(hipError_t e) { return last_error = e; }
}  // namespace

extern "C" {
hipError_t hipGetDevice(int* d) { *d = 0; return hipSuccess; }
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipGetLastError() { const hipError_t e = last_error; last_error = hipSuccess; return e; }
const char* hipGetErrorString(hipError_t) { return "error"; }
hipError_t hipDeviceSynchronize() {
    if (capturing) return fail_with(hipErrorStreamCaptureUnsupported);
    ++waits;
    return hipSuccess;
}
hipError_t hipMalloc(void** p, size_t n) {
    if (capturing) return fail_with(hipErrorStreamCaptureUnsupported);
    last_size = n;
    if (total + n > limit) return fail_with(hipErrorOutOfMemory);
    *p = reinterpret_cast<void*>(next_address += 4096);
    allocated[*p] = n;
    total += n;
    return hipSuccess;
}
hipError_t hipFree(void* p) {
    if (capturing) return fail_with(hipErrorStreamCaptureUnsupported);
    ++frees;
    total -= allocated.at(p);
    allocated.erase(p);
    return hipSuccess;
}
hipError_t hipStreamIsCapturing(hipStream_t, hipStreamCaptureStatus* s) {
    *s = capturing ? hipStreamCaptureStatusActive : hipStreamCaptureStatusNone;
    return hipSuccess;
}
hipError_t hipMemcpy(void*, const void*, size_t, hipMemcpyKind) { return hipSuccess; }
}

#define CHECK(x)                                                     \
    do {                                                             \
        if (!(x)) {                                                  \
            std::printf("line %d: %s\n", __LINE__, #x);              \
            return 1;                                                \
        }                                                            \
    } while (0)

int main() {
    constexpr size_t kMiB = size_t(1) << 20, kGiB = size_t(1) << 30;
    using ra::DeviceBuffer;
    {  // Reuse: a block that may be in use is waited for first, an idle one is not.
        DeviceBuffer a, b;
        CHECK(a.allocate(10 * kMiB) == RA_OK);
        void* p = a.get();
        a.reset();
        CHECK(waits == 0);
        CHECK(a.allocate(10 * kMiB) == RA_OK && a.get() == p && waits == 1);
        a.reset_idle();
        CHECK(b.allocate(9 * kMiB) == RA_OK && b.get() == p && waits == 1);
        b.reset();
        CHECK(a.allocate(20 * kMiB) == RA_OK && a.get() != p && waits == 1);  // does not fit: no wait for it
    }
    ra::pool_trim();
    CHECK(total == 0 && frees == 2);
    {  // Capture: giving back calls nothing, and nothing is handed on before it ends.
        DeviceBuffer a, b, grown;
        CHECK(a.allocate(10 * kMiB) == RA_OK && grown.ensure(kMiB, nullptr) == RA_OK);
        CHECK(b.allocate(10 * kMiB) == RA_OK);
        void *p = a.get(), *q = b.get();
        b.reset_idle();
        waits = 0;
        capturing = true;
        a.reset();
        CHECK(last_error == hipSuccess);
        CHECK(a.allocate(10 * kMiB) == RA_OK && a.get() == q);  // idle since before
        CHECK(b.allocate(10 * kMiB) != RA_OK && b.get() == nullptr);
        CHECK(last_error == hipErrorStreamCaptureUnsupported || last_error == hipSuccess);
        last_error = hipSuccess;
        a.reset_idle();
        CHECK(grown.ensure(10 * kMiB, nullptr) != RA_OK);  // refused whatever the pool holds
        last_error = hipSuccess;
        capturing = false;
        CHECK(grown.ensure(10 * kMiB, nullptr) == RA_OK && grown.get() == q);
        CHECK(b.allocate(10 * kMiB) == RA_OK && b.get() == p && waits == 1);
    }
    ra::pool_trim();
    CHECK(total == 0 && allocated.empty());
    {  // Bound: the oldest blocks go back, at the end all of them.
        DeviceBuffer v[6];
        for (auto& x : v) CHECK(x.allocate(kGiB) == RA_OK);
        void* newest = v[5].get();
        for (auto& x : v) x.reset();
        CHECK(total == ra::kPoolBytes);
        CHECK(allocated.count(newest) == 1);
        // A full pool cannot free under capture: it keeps the block and leaves no error.
        DeviceBuffer w;
        CHECK(w.allocate(3 * kGiB) == RA_OK);
        capturing = true;
        w.reset();
        CHECK(last_error == hipSuccess && total == ra::kPoolBytes + 3 * kGiB);
        capturing = false;
        DeviceBuffer t;
        CHECK(t.allocate(kMiB) == RA_OK);
        t.reset();
        CHECK(total <= ra::kPoolBytes);
    }
    ra::pool_trim();
    CHECK(total == 0);
    {  // Sizes: rounded up by an eighth at most, not where the pool would not keep it or nothing else fits.
        DeviceBuffer a;
        CHECK(a.allocate(1000 * kMiB + 1) == RA_OK && last_size > 1000 * kMiB && last_size <= 1125 * kMiB + 1);
        CHECK(a.allocate(5 * kGiB + 4096) == RA_OK && last_size == 5 * kGiB + 4096);
        a.reset();
        limit = 3 * kGiB + 64 * kMiB;
        CHECK(a.allocate(3 * kGiB + 32 * kMiB) == RA_OK && last_size == 3 * kGiB + 32 * kMiB && a.bytes() == last_size);
        CHECK(a.allocate(3 * kGiB + 65 * kMiB) == RA_ERR_OUT_OF_MEMORY && a.get() == nullptr && a.bytes() == 0);
        CHECK(a.allocate(3 * kGiB) == RA_OK);
    }
    std::printf("pool ok\n");
    return 0;
}

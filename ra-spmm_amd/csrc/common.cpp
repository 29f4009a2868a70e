// common.cpp — error state, names, the host parallel_for and the device memory
// pool of the C ABI.
#include <algorithm>
#include <atomic>
#include <map>
#include <mutex>
#include <thread>

#include "ra_internal.hpp"

namespace ra {

namespace {
thread_local std::string g_last_error;
}

void set_error(const std::string& msg) { g_last_error = msg; }
void clear_error() { g_last_error.clear(); }

void parallel_for(int64_t n, int64_t grain, const std::function<void(int64_t, int64_t)>& f) {
    if (n <= 0) return;
    grain = std::max<int64_t>(1, grain);
    const int64_t chunks = (n + grain - 1) / grain;
    unsigned hw = std::thread::hardware_concurrency();
    if (hw == 0) hw = 1;
    const int64_t nthreads = std::min<int64_t>(std::min<int64_t>(hw, 64), chunks);
    if (nthreads <= 1) {
        f(0, n);
        return;
    }
    std::atomic<int64_t> next{0};
    auto worker = [&]() {
        for (;;) {
            const int64_t c = next.fetch_add(1);
            if (c >= chunks) break;
            const int64_t b = c * grain;
            f(b, std::min(n, b + grain));
        }
    };
    std::vector<std::thread> pool;
    pool.reserve(nthreads - 1);
    for (int64_t t = 1; t < nthreads; ++t) pool.emplace_back(worker);
    worker();
    for (auto& t : pool) t.join();
}

// ------------------------------------------------------- device memory pool
namespace {

struct PoolBlock {
    void* ptr;
    uint64_t age;
};

struct DevicePool {
    std::multimap<size_t, PoolBlock> free_blocks;  // by capacity
    // Given back while the device may still be using them: free once it has
    // been waited for, which the first request that could use one does.
    std::multimap<size_t, PoolBlock> pending;
    size_t held = 0;  // bytes of both
};

struct Pool {
    std::mutex mutex;
    std::map<int, DevicePool> devices;
    uint64_t clock = 0;
};

// Never destroyed: plans may outlive static destructors, and the runtime frees
// the memory at exit.
Pool& pool() {
    static Pool* p = new Pool();
    return *p;
}

// Eight classes per power of two, so that plans of graphs of about the same size
// use each other's blocks; a class is at most 1/8 over the request, and a kept
// block at most 1/4 over its class (take).  What the pool never keeps is not
// rounded.
size_t size_class(size_t bytes) {
    if (bytes > kPoolBytes) return bytes;
    size_t power = 4096;
    while (power * 2 <= bytes) power *= 2;
    const size_t step = power / 8;
    return (bytes + step - 1) / step * step;
}

// Current device switched for one scope.
class OnDevice {
public:
    explicit OnDevice(int device) {
        (void)hipGetDevice(&old_);
        if (old_ != device) (void)hipSetDevice(device);
        switched_ = old_ != device;
    }
    ~OnDevice() {
        if (switched_) (void)hipSetDevice(old_);
    }

private:
    int old_ = 0;
    bool switched_ = false;
};

// hipFree, which waits for the device by itself.  Its error (a stream is being
// captured) is not left for the next launch check.
bool free_block(void* ptr) {
    if (hipFree(ptr) == hipSuccess) return true;
    (void)hipGetLastError();
    return false;
}

// Free the blocks of `d` from the oldest on until at most `keep` bytes are held,
// or until one cannot be freed now.
void trim_locked(int device, DevicePool& d, size_t keep) {
    if (d.held <= keep) return;
    const OnDevice on(device);
    while (d.held > keep) {
        std::multimap<size_t, PoolBlock>* list = nullptr;
        std::multimap<size_t, PoolBlock>::iterator oldest;
        for (auto* l : {&d.free_blocks, &d.pending})
            for (auto it = l->begin(); it != l->end(); ++it)
                if (!list || it->second.age < oldest->second.age) {
                    list = l;
                    oldest = it;
                }
        if (!list || !free_block(oldest->second.ptr)) return;
        d.held -= oldest->first;
        list->erase(oldest);
    }
}

// A kept block of `want` bytes or a quarter more, or the end of the list.
std::multimap<size_t, PoolBlock>::iterator find_block(std::multimap<size_t, PoolBlock>& list, size_t want) {
    const auto it = list.lower_bound(want);
    return it != list.end() && it->first <= want + want / 4 ? it : list.end();
}

bool take(DevicePool& d, size_t want, void** ptr, size_t* capacity) {
    const auto it = find_block(d.free_blocks, want);
    if (it == d.free_blocks.end()) return false;
    *ptr = it->second.ptr;
    *capacity = it->first;
    d.held -= it->first;
    d.free_blocks.erase(it);
    return true;
}

}  // namespace

ra_status pool_allocate(void** ptr, size_t bytes, bool kept, size_t* capacity, int* device) {
    *ptr = nullptr;
    RA_HIP_TRY(hipGetDevice(device));
    const size_t want = kept ? size_class(bytes) : bytes;
    Pool& p = pool();
    if (kept) {
        std::multimap<size_t, PoolBlock> waited;
        {
            std::lock_guard<std::mutex> lock(p.mutex);
            DevicePool& d = p.devices[*device];
            if (take(d, want, ptr, capacity)) return RA_OK;
            if (find_block(d.pending, want) != d.pending.end()) waited.swap(d.pending);
        }
        if (!waited.empty()) {
            const bool idle = hipDeviceSynchronize() == hipSuccess;
            if (!idle) (void)hipGetLastError();  // a stream is being captured: they stay pending
            std::lock_guard<std::mutex> lock(p.mutex);
            DevicePool& d = p.devices[*device];
            (idle ? d.free_blocks : d.pending).merge(waited);
            if (idle && take(d, want, ptr, capacity)) return RA_OK;
        }
    }
    size_t size = want;
    hipError_t e = hipMalloc(ptr, size);
    if (e == hipErrorOutOfMemory) {
        (void)hipGetLastError();
        {
            std::lock_guard<std::mutex> lock(p.mutex);
            trim_locked(*device, p.devices[*device], 0);
        }
        size = bytes;  // no more than was asked for
        e = hipMalloc(ptr, size);
    }
    if (e != hipSuccess) {
        *ptr = nullptr;
        return hip_fail(e, "hipMalloc");
    }
    *capacity = size;
    return RA_OK;
}

void pool_release(void* ptr, size_t capacity, int device, bool idle) {
    if (capacity > kPoolBytes) {
        const OnDevice on(device);
        (void)free_block(ptr);
        return;
    }
    Pool& p = pool();
    std::lock_guard<std::mutex> lock(p.mutex);
    DevicePool& d = p.devices[device];
    (idle ? d.free_blocks : d.pending).emplace(capacity, PoolBlock{ptr, ++p.clock});
    d.held += capacity;
    trim_locked(device, d, kPoolBytes);
}

void pool_trim() {
    Pool& p = pool();
    std::lock_guard<std::mutex> lock(p.mutex);
    for (auto& d : p.devices) trim_locked(d.first, d.second, 0);
}

}  // namespace ra

extern "C" {

void ra_release_memory(void) { ra::pool_trim(); }

int ra_abi_version(void) { return RA_SPMM_ABI_VERSION; }

const char* ra_last_error(void) { return ra::g_last_error.c_str(); }

const char* ra_status_string(ra_status s) {
    switch (s) {
        case RA_OK: return "RA_OK";
        case RA_ERR_INVALID_ARGUMENT: return "RA_ERR_INVALID_ARGUMENT";
        case RA_ERR_HIP: return "RA_ERR_HIP";
        case RA_ERR_OUT_OF_MEMORY: return "RA_ERR_OUT_OF_MEMORY";
        case RA_ERR_UNSUPPORTED: return "RA_ERR_UNSUPPORTED";
        case RA_ERR_INACTIVE_PLAN: return "RA_ERR_INACTIVE_PLAN";
        case RA_ERR_INTERNAL: return "RA_ERR_INTERNAL";
    }
    return "RA_ERR_UNKNOWN";
}

// Path names keep the reference spelling (ra_common.h:116-135) because the
// router dict, the Python mirror and the harness labels all key on them.
const char* ra_path_name(int32_t p) {
    static const char* const kNames[RA_PATH_COUNT] = {
        "CSR_DIRECT",   "CSR_ADAPTIVE",      "STAGED_REUSE",   "TC_SPARSE",
        "ROW_SPLIT_CUDA", "TC_REORDERED",    "HYBRID_TC_CUDA", "CUSPARSE",
        "RODE_ENHANCED", "VECTORIZED_COARSE", "LOCALITY_TILED", "TC_DIRECT",
        "COMMUNITY_TC", "ZERO_OVERHEAD_CSR", "SEGMENT_HYBRID"};
    if (p < 0 || p >= RA_PATH_COUNT) return "UNKNOWN";
    return kNames[p];
}

// Rejection names keep the reference spelling (ra_common.h:161-178).
const char* ra_reject_name(int32_t c) {
    static const char* const kNames[] = {
        "CHOSEN",         "NOT_FEASIBLE",     "LOW_FILL",          "LOW_COVERAGE",
        "HIGH_SKEW",      "SMALL_N",          "INSUFFICIENT_NNZ",  "LOW_OCCUPANCY",
        "LOW_DEGREE_SKEW", "NOT_STRONG_ENOUGH", "MARGIN_TOO_SMALL", "NOT_IN_PORTFOLIO",
        "UNKNOWN"};
    if (c < 0 || c > RA_REJECT_UNKNOWN) return "UNKNOWN";
    return kNames[c];
}

}  // extern "C"

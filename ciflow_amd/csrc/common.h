// Shared definitions for the ciflow_amd library (host + device).
#pragma once

#include <hip/hip_runtime.h>

#include "block_cache.h"
#include "errors.h"

#include <chrono>
#include <cstdint>
#include <cstdio>
#include <memory>
#include <stdexcept>
#include <string>
#include <vector>

namespace cf {

typedef uint64_t str_t;  // one spin string: bit k = spatial orbital k occupied

#define CF_HIP(call)                                                                          \
    do {                                                                                      \
        hipError_t e_ = (call);                                                               \
        if (e_ != hipSuccess)                                                                 \
            throw ::cf::Error(e_ == hipErrorOutOfMemory ? ::cf::ERR_NOMEM : ::cf::ERR_HIP,    \
                              std::string(#call) + ": " + hipGetErrorString(e_));             \
    } while (0)

// A context's blocks: from and back to the device in its stream's order.
struct HipBlockSource : BlockSource {
    hipStream_t stream;
    explicit HipBlockSource(hipStream_t s) : stream(s) {}
    void* alloc(size_t bytes) override {
        void* p = nullptr;
        const hipError_t e = hipMallocAsync(&p, bytes, stream);
        if (e == hipSuccess) return p;
        (void)hipGetLastError();
        if (e == hipErrorOutOfMemory) return nullptr;
        throw Error(ERR_HIP, std::string("hipMallocAsync: ") + hipGetErrorString(e));
    }
    void free(void* p) override { (void)hipFreeAsync(p, stream); }
    void free_unordered(void* p) override { (void)hipFree(p); }
    void drain() override { (void)hipStreamSynchronize(stream); }
    // less than an eighth of the device free (kept blocks count as used), asked for
    // every 10 ms at most: 4 us a call, which a matrix build would make ten times
    bool scarce() override {
        const auto now = std::chrono::steady_clock::now();
        if (now < next_look) return is_scarce;
        size_t free_b = 0, total_b = 0;
        if (hipMemGetInfo(&free_b, &total_b) != hipSuccess) {
            (void)hipGetLastError();
            return false;
        }
        next_look = now + std::chrono::milliseconds(10);
        return is_scarce = free_b < total_b / 8;
    }

  private:  // read and written under the cache's lock
    std::chrono::steady_clock::time_point next_look{};
    bool is_scarce = false;
};
struct DeviceBlocks {
    HipBlockSource src;
    BlockCache cache;
    DeviceBlocks(hipStream_t s, BlockBudget* b) : src(s), cache(&src, b) {}
};

// The blocks that device buffers allocated on this host thread come from: a
// context makes its own current here, so allocating and freeing neither
// blocks the host nor waits for other streams.  Null: plain hipMalloc / hipFree.
inline thread_local std::shared_ptr<DeviceBlocks> tls_blocks;

// The device's block caches and what they may keep together (1/16 of its memory).
BlockBudget* block_budget(int device);

// hipMalloc for memory outside of the caches: one that fails takes back what they keep.
inline void* device_malloc(size_t bytes) {
    void* p = nullptr;
    hipError_t e = hipMalloc(&p, bytes);
    if (e == hipErrorOutOfMemory) {
        (void)hipGetLastError();
        int device = 0;
        CF_HIP(hipGetDevice(&device));
        block_budget(device)->trim_all();
        e = hipMalloc(&p, bytes);
    }
    if (e == hipSuccess) return p;
    (void)hipGetLastError();
    if (e == hipErrorOutOfMemory) throw Error(ERR_NOMEM, "device memory: " + std::to_string(bytes) + " bytes");
    throw Error(ERR_HIP, std::string("hipMalloc: ") + hipGetErrorString(e));
}

// Owning device buffer.
template <class T>
struct DBuf {
    T* p = nullptr;
    size_t n = 0;
    size_t block = 0;                 // bytes of the block it holds
    std::shared_ptr<DeviceBlocks> s;  // where it came from (null: hipMalloc)
    DBuf() = default;
    explicit DBuf(size_t count) { alloc(count); }
    DBuf(const DBuf&) = delete;
    DBuf& operator=(const DBuf&) = delete;
    DBuf(DBuf&& o) noexcept { swap(o); }
    DBuf& operator=(DBuf&& o) noexcept {
        if (this != &o) {
            release();
            swap(o);
        }
        return *this;
    }
    ~DBuf() { release(); }
    void swap(DBuf& o) noexcept {
        std::swap(p, o.p);
        std::swap(n, o.n);
        std::swap(block, o.block);
        std::swap(s, o.s);
    }
    void alloc(size_t count) {
        release();
        if (count) {
            if (tls_blocks) {
                p = (T*)tls_blocks->cache.take(count * sizeof(T), &block);
                if (!p) throw Error(ERR_NOMEM, "device memory: " + std::to_string(count * sizeof(T)) + " bytes");
                s = tls_blocks;
            } else {
                p = (T*)device_malloc(count * sizeof(T));
            }
        }
        n = count;
    }
    void release() {
        if (p) {
            if (s) s->cache.give(p, block);
            else (void)hipFree(p);
        }
        p = nullptr;
        n = 0;
        block = 0;
        s.reset();
    }
    size_t bytes() const { return n * sizeof(T); }
};

// Binomial coefficients C(k, m) for 0 <= k <= 64, 0 <= m <= 64 (exact while < 2^64).
inline uint64_t binom_host(int n, int k) {
    if (k < 0 || k > n) return 0;
    unsigned __int128 r = 1;
    for (int i = 1; i <= k; ++i) r = r * (unsigned)(n - k + i) / (unsigned)i;
    return (uint64_t)r;
}


}  // namespace cf

// Shared definitions for the ciflow_amd library (host + device).
#pragma once

#include <hip/hip_runtime.h>

#include "block_cache.h"
#include "errors.h"

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
                CF_HIP(hipMalloc((void**)&p, count * sizeof(T)));
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

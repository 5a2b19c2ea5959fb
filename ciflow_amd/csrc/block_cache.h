// Device blocks kept for reuse, one cache per context (stream).
//
// The runtime's stream-ordered pool gives freed memory back at once whatever
// its release threshold says (its reserved size is 0 right after a
// hipFreeAsync, on the default pool and on pools of our own), so every call
// paid for mapping and unmapping its device memory: 0.2 ms per block above
// 100 MB in a fresh process and far more in one that has held other matrices.
// Measured on MI355X, a pass before / with the blocks kept: build of an FCI
// L=11 5a4b matrix and its first product 100.8 / 6.4 ms (6.3 ms of kernels when
// introduced), matrix of a 95,040-determinant list and its first product
// 171 / 15.0 ms, 12 DOCI L=19 solves 27.3 / 20.3 ms, an FCI L=11 2-RDM
// 12.6 / 3.2 ms.
//
// Blocks given back here are handed out again only by the same cache, that is
// to work on the same stream, so reuse needs no wait: what still reads or
// writes a block was enqueued before what gets it next.  The bytes kept are
// bounded over all caches of a device; a block past the bound pushes out the
// cache's oldest ones or goes back itself, one that was not reused for
// kKeepTakes requests goes back, an allocation that fails first takes back
// what every cache of the device holds, and close() returns the rest.  What other
// libraries and processes on the device need is not seen here: a large block is
// not kept while the device is short of memory, and cf_ctx_trim gives back all.
//
// No HIP in this file: the policy is tested on the CPU with a source of its own.
#pragma once

#include <algorithm>
#include <cstddef>
#include <cstdint>
#include <iterator>
#include <list>
#include <map>
#include <mutex>
#include <new>
#include <vector>

namespace cf {

// Where blocks come from and go back to.
struct BlockSource {
    virtual ~BlockSource() = default;
    virtual void* alloc(size_t bytes) = 0;        // nullptr: no memory
    virtual void free(void* p) = 0;               // after the work enqueued so far
    virtual void free_unordered(void* p) = 0;     // once the owner (its stream) is gone
    virtual void drain() = 0;                     // until freed blocks are really back
    virtual bool scarce() { return false; }       // others of the device may need a block more than we do
};

class BlockCache;

// The caches of one device and the bytes that they may keep together.
struct BlockBudget {
    std::mutex mu;  // taken before a cache's own
    uint64_t limit = 0, cached = 0;
    std::vector<BlockCache*> caches;
    std::mutex cached_mu;
    bool reserve(uint64_t b) {
        std::lock_guard<std::mutex> lk(cached_mu);
        if (cached + b > limit) return false;
        cached += b;
        return true;
    }
    void unreserve(uint64_t b) {
        std::lock_guard<std::mutex> lk(cached_mu);
        cached -= b;
    }
    uint64_t held() {
        std::lock_guard<std::mutex> lk(cached_mu);
        return cached;
    }
    inline uint64_t trim_all();  // bytes given back
};

class BlockCache {
  public:
    static constexpr uint64_t kKeepTakes = 4096;
    static constexpr size_t kLarge = 32u << 20;  // blocks worth a look at the device's free memory

    BlockCache(BlockSource* src, BlockBudget* budget) : src_(src), budget_(budget) {
        std::lock_guard<std::mutex> lk(budget_->mu);
        budget_->caches.push_back(this);
    }
    ~BlockCache() { close(); }
    BlockCache(const BlockCache&) = delete;
    BlockCache& operator=(const BlockCache&) = delete;

    // A block of at least `bytes` (> 0); *got is its size, to be given back with it.
    void* take(size_t bytes, size_t* got) {
        const size_t want = (bytes + 255) / 256 * 256;
        {
            std::lock_guard<std::mutex> lk(mu_);
            ++takes_;
            auto it = by_size_.lower_bound(want);
            if (it != by_size_.end() && it->first <= most(want)) {
                void* p = it->second->p;
                *got = it->first;
                forget(it);
                return p;
            }
        }
        void* p = src_->alloc(want);
        if (!p) {
            budget_->trim_all();
            p = src_->alloc(want);
        }
        *got = want;
        return p;
    }

    void give(void* p, size_t bytes) noexcept {
        std::lock_guard<std::mutex> lk(mu_);  // held throughout: close() waits before the stream goes
        if (closed_) {
            src_->free_unordered(p);
            return;
        }
        while (!age_.empty() && takes_ - age_.front().take > kKeepTakes) src_->free(evict());
        if (bytes >= kLarge && src_->scarce()) {
            src_->free(p);
            return;
        }
        bool kept = budget_->reserve(bytes);
        while (!kept && bytes <= budget_->limit && !age_.empty()) {
            src_->free(evict());
            kept = budget_->reserve(bytes);
        }
        if (kept) {
            bool listed = false;
            try {
                age_.push_back(Block{p, bytes, takes_});
                listed = true;
                by_size_.emplace(bytes, std::prev(age_.end()));
                return;
            } catch (const std::bad_alloc&) {
                if (listed) age_.pop_back();
                budget_->unreserve(bytes);
            }
        }
        src_->free(p);
    }

    // Every kept block goes back; their bytes.
    uint64_t trim() {
        std::lock_guard<std::mutex> lk(mu_);
        uint64_t bytes = 0;
        while (!age_.empty()) {
            bytes += age_.front().bytes;
            src_->free(evict());
        }
        return bytes;
    }

    // Every kept block goes back, and blocks given later go straight back.
    void close() {
        {
            std::lock_guard<std::mutex> lk(budget_->mu);
            auto& v = budget_->caches;
            v.erase(std::remove(v.begin(), v.end(), this), v.end());
        }
        std::lock_guard<std::mutex> lk(mu_);
        while (!age_.empty()) src_->free(evict());
        closed_ = true;
    }

    void drain() { src_->drain(); }

  private:
    struct Block {
        void* p;
        size_t bytes;
        uint64_t take;  // takes_ when it was given back
    };
    typedef std::multimap<size_t, std::list<Block>::iterator> SizeMap;

    // The largest block that serves a request of `want` bytes: small ones up to
    // twice as large, large ones hardly larger than asked for, since what a live
    // buffer wastes cannot be taken back.
    static size_t most(size_t want) {
        if (want <= (64u << 10)) return 2 * want;
        if (want <= (64u << 20)) return want + want / 8;
        return want + want / 64;
    }
    void forget(SizeMap::iterator it) {
        budget_->unreserve(it->first);
        age_.erase(it->second);
        by_size_.erase(it);
    }
    void* evict() {  // the block kept longest
        auto first = age_.begin();
        void* p = first->p;
        auto it = by_size_.lower_bound(first->bytes);
        while (it->second != first) ++it;
        forget(it);
        return p;
    }

    std::mutex mu_;
    BlockSource* src_;
    BlockBudget* budget_;
    std::list<Block> age_;  // oldest first
    SizeMap by_size_;
    uint64_t takes_ = 0;
    bool closed_ = false;
};

inline uint64_t BlockBudget::trim_all() {
    std::lock_guard<std::mutex> lk(mu);
    uint64_t bytes = 0;
    for (BlockCache* c : caches) {
        bytes += c->trim();
        c->drain();
    }
    return bytes;
}

}  // namespace cf

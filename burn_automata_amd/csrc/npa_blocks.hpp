// npa_blocks.hpp - device memory: allocation, and the blocks that destroyed states leave for the next ones.
#pragma once

#include <stddef.h>

#include <algorithm>
#include <mutex>
#include <vector>

namespace npa {

// Device blocks of one context's destroyed states: a rollout of 64 x 4,096 particles spent more time in the
// allocation and release of its 118 MB state than in 16 steps (6.0 ms a call, 2.8 ms of it kernels).
// Bounded (kBlocks blocks, kBytes in all; the block kept longest goes first), locked because states may be
// destroyed on any thread, and given back with the pool, by clear(), and wherever an allocation of this library,
// through whichever context, finds no memory left (allocate()).
//
// Mem: Error; Error alloc(void**, size_t); void free(void*); bool ok(Error), out_of_memory(Error).
template <class Mem>
class BlockPool {
  public:
    struct Block {
        void* ptr = nullptr;
        size_t bytes = 0;
    };
    using Error = typename Mem::Error;
    static constexpr size_t kBlocks = 4, kBytes = (size_t)1 << 30, kGrain = (size_t)2 << 20;

    BlockPool() {
        std::lock_guard<std::mutex> lock(pools().mutex);
        pools().all.push_back(this);
    }
    ~BlockPool() {
        {
            std::lock_guard<std::mutex> lock(pools().mutex);
            auto& all = pools().all;
            all.erase(std::find(all.begin(), all.end(), this));
        }
        clear();
    }
    BlockPool(const BlockPool&) = delete;
    BlockPool& operator=(const BlockPool&) = delete;

    // Device memory; when there is none left, the kept blocks of every pool are given back first.
    static Error allocate(void** ptr, size_t bytes) {
        Error e = Mem::alloc(ptr, bytes);
        if (!Mem::out_of_memory(e)) return e;
        {
            std::lock_guard<std::mutex> lock(pools().mutex);
            for (BlockPool* p : pools().all) p->clear();
        }
        return Mem::alloc(ptr, bytes);
    }

    // The smallest kept block that fits without wasting more than its need again, else a new one.
    Error acquire(size_t bytes, Block* out) {
        const size_t want = (bytes + kGrain - 1) / kGrain * kGrain;
        {
            std::lock_guard<std::mutex> lock(mutex_);
            size_t best = kept_.size();
            for (size_t k = 0; k < kept_.size(); ++k)
                if (kept_[k].bytes >= want && kept_[k].bytes <= 2 * want && (best == kept_.size() || kept_[k].bytes < kept_[best].bytes))
                    best = k;
            if (best < kept_.size()) {
                *out = kept_[best];
                kept_.erase(kept_.begin() + (ptrdiff_t)best);
                return Error();
            }
        }
        Block b{nullptr, want};
        const Error e = allocate(&b.ptr, want);
        *out = Mem::ok(e) ? b : Block();
        return e;
    }

    // Keeps the block for the next acquire; no queued work may use it any more.
    void release(Block b) {
        if (!b.ptr) return;
        std::vector<Block> gone;
        {
            std::lock_guard<std::mutex> lock(mutex_);
            if (b.bytes > kBytes) {
                gone.push_back(b);
            } else {
                size_t total = b.bytes;
                for (const Block& k : kept_) total += k.bytes;
                while (kept_.size() >= kBlocks || total > kBytes) {  // the oldest: sizes no longer asked for leave
                    total -= kept_.front().bytes;
                    gone.push_back(kept_.front());
                    kept_.erase(kept_.begin());
                }
                kept_.push_back(b);
            }
        }
        for (const Block& g : gone) Mem::free(g.ptr);
    }

    void clear() {
        std::vector<Block> gone;
        {
            std::lock_guard<std::mutex> lock(mutex_);
            gone.swap(kept_);
        }
        for (const Block& g : gone) Mem::free(g.ptr);
    }

  private:
    struct Pools {
        std::mutex mutex;
        std::vector<BlockPool*> all;
    };
    static Pools& pools() {
        static Pools* p = new Pools;  // contexts may outlive static destruction
        return *p;
    }
    std::mutex mutex_;
    std::vector<Block> kept_;
};

}  // namespace npa

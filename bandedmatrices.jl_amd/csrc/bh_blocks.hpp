// bh_blocks.hpp -- the large device blocks that bh_free keeps for bh_malloc.
//
// Mapping and unmapping one costs far more than the work of many calls
// (hipMalloc + hipFree: 4 us at 2 MB, 28 at 16 MB, 280 at 69-103 MB), and a
// program that factors in a loop frees what it is about to ask for.  So a
// freed block of at least kMin bytes is kept, up to kKeep bytes in all, after
// waiting for the device as hipFree does (no work of any stream can still
// touch a kept block); the oldest go back when there is no room, those not
// asked for over kAge frees, and all of them when the device runs out.
//
// The bookkeeping only, without HIP's headers: Dev supplies the runtime (its
// calls return 0 or an error code), so that it can be tested on the host.
//   int current(int *dev)            the calling thread's device
//   int alloc(void **p, size_t n), release(void *p), wait()
//   void others()                    gives back what else is kept (the device ran out)
//   static constexpr int kNoMemory, kBadPointer
#pragma once
#include <stddef.h>

#include <mutex>
#include <unordered_map>
#include <vector>

namespace bh {

template <class Dev>
class BlockCache {
  public:
    static constexpr size_t kMin = size_t(8) << 20;
    static constexpr size_t kKeep = size_t(1) << 30;
    static constexpr unsigned long long kAge = 64;

    explicit BlockCache(Dev dev = Dev()) : dev_(dev) {}

    int take(void **p, size_t bytes) {
        int d = -1;
        std::unique_lock<std::mutex> lock(m_, std::defer_lock);
        const bool track = bytes >= kMin && dev_.current(&d) == 0;
        if (!track) {
            int e = dev_.alloc(p, bytes);
            if (e != Dev::kNoMemory) return e;
            drop();
            dev_.others();
            return dev_.alloc(p, bytes);
        }
        lock.lock();
        size_t best = kept_.size();
        for (size_t i = 0; i < kept_.size(); ++i)
            if (kept_[i].dev == d && kept_[i].bytes >= bytes && kept_[i].bytes <= bytes + bytes / 8 &&
                (best == kept_.size() || kept_[i].bytes < kept_[best].bytes))
                best = i;
        if (best < kept_.size()) {
            *p = kept_[best].p;
            kept_bytes_ -= kept_[best].bytes;
            used_[*p] = kept_[best];
            kept_.erase(kept_.begin() + best);
            return 0;
        }
        int e = dev_.alloc(p, bytes);
        if (e == Dev::kNoMemory) {
            trim(0, kKeep);
            dev_.others();
            e = dev_.alloc(p, bytes);
        }
        if (e == 0) used_[*p] = Block{*p, bytes, d, 0, false};
        return e;
    }

    int give(void *p) {
        int d = -1;
        std::unique_lock<std::mutex> lock(m_);
        const auto it = used_.find(p);
        if (it == used_.end()) {
            // a block kept here is the runtime's still: it would free it once
            // more, and the next take would hand out unmapped memory
            for (const Block &b : kept_)
                if (b.p == p) return Dev::kBadPointer;
            lock.unlock();
            return dev_.release(p);
        }
        if (it->second.leaving) return Dev::kBadPointer;  // another thread frees it now
        ++clock_;
        Block b = it->second;
        if (b.bytes > kKeep / 2 || dev_.current(&d) != 0 || d != b.dev) {
            used_.erase(it);
            lock.unlock();
            return dev_.release(p);
        }
        it->second.leaving = true;
        lock.unlock();
        const int e = dev_.wait();  // what a free waits for
        lock.lock();
        if (e != 0) {  // nothing is freed: the caller may try again
            used_[p].leaving = false;
            return e;
        }
        used_.erase(p);
        trim(kAge, b.bytes);
        b.at = clock_;
        b.leaving = false;
        kept_.push_back(b);
        kept_bytes_ += b.bytes;
        return 0;
    }

    // Give back every kept block.
    void drop() {
        std::lock_guard<std::mutex> lock(m_);
        trim(0, kKeep);
    }

    size_t kept_bytes() {
        std::lock_guard<std::mutex> lock(m_);
        return kept_bytes_;
    }

  private:
    struct Block {
        void *p;
        size_t bytes;
        int dev;
        unsigned long long at;  // the clock when it was freed
        bool leaving;           // its free waits for the device
    };

    // Give back the kept blocks past `age` frees, then the oldest until `bytes`
    // more fit.  The mutex is held.
    void trim(unsigned long long age, size_t bytes) {
        size_t i = 0;
        while (i < kept_.size() && (clock_ - kept_[i].at > age || kept_bytes_ + bytes > kKeep)) {
            (void)dev_.release(kept_[i].p);
            kept_bytes_ -= kept_[i].bytes;
            ++i;
        }
        kept_.erase(kept_.begin(), kept_.begin() + i);
    }

    Dev dev_;
    std::mutex m_;
    std::unordered_map<void *, Block> used_;
    std::vector<Block> kept_;  // oldest first
    size_t kept_bytes_ = 0;
    unsigned long long clock_ = 0;
};

}  // namespace bh

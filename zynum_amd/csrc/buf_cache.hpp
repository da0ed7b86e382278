// Cache of idle buffers: what a call gives back the next call takes again
// instead of allocating.
#pragma once

#include <stddef.h>

#include <mutex>
#include <vector>

namespace zg {

// Memory: alloc(bytes) (null on failure), free(p), and place(), the number of
// the place the calling thread's buffers live in (its current device).  A
// buffer is handed only to callers of the place it was allocated in, and to
// any request it holds with at most twice the size.  Up to `cap` bytes are
// kept idle, over all places.
template <class Memory>
class BufCache {
  public:
    explicit BufCache(size_t cap, Memory memory = Memory()) : memory_(memory), cap_(cap) {}

    void* acquire(size_t bytes, size_t* got) {
        const int place = memory_.place();
        {
            std::lock_guard<std::mutex> lock(mu_);
            size_t best = free_.size();
            for (size_t i = 0; i < free_.size(); ++i) {
                const size_t b = free_[i].bytes;
                if (free_[i].place == place && b >= bytes && b <= 2 * bytes + kGranule &&
                    (best == free_.size() || b < free_[best].bytes))
                    best = i;
            }
            if (best < free_.size()) {
                const Buf buf = free_[best];
                free_.erase(free_.begin() + (ptrdiff_t)best);
                cached_ -= buf.bytes;
                *got = buf.bytes;
                return buf.ptr;
            }
        }
        const size_t want = (bytes + kGranule - 1) / kGranule * kGranule;
        void* p = memory_.alloc(want);
        if (p != nullptr) *got = want;
        return p;
    }

    // In the place it was acquired in; the caller has synchronised the stream
    // that used the buffer.
    void release(void* p, size_t bytes) {
        const int place = memory_.place();
        {
            std::lock_guard<std::mutex> lock(mu_);
            if (cached_ + bytes <= cap_) {
                free_.push_back({p, bytes, place});
                cached_ += bytes;
                return;
            }
        }
        memory_.free(p);
    }

    void free_all() {
        std::lock_guard<std::mutex> lock(mu_);
        for (const Buf& b : free_) memory_.free(b.ptr);
        free_.clear();
        cached_ = 0;
    }

  private:
    struct Buf {
        void* ptr;
        size_t bytes;
        int place;
    };
    static constexpr size_t kGranule = size_t(2) << 20;
    Memory memory_;
    size_t cap_;
    std::mutex mu_;
    std::vector<Buf> free_;
    size_t cached_ = 0;
};

}  // namespace zg

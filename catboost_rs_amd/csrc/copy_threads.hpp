// Host threads that copy a table chunk by chunk while the caller passes the finished chunks on.
#pragma once
#include <atomic>
#include <cstdint>
#include <thread>
#include <vector>

namespace cbh {

// copy(chunk, first, step) copies the features first, first + step, ... of a chunk.  Chunk c may be
// filled once `open` has passed it; `done[c]` counts the threads that have copied their features of
// it.  Threads that cannot be started, for whatever reason, are done without: those there take all
// of it, the caller if there is none.  The destructor ends and joins them wherever they are, so an
// exception on the caller's side leaves no thread behind.
template <class Copy>
class CopyThreads {
  public:
    CopyThreads(unsigned want, uint64_t n_chunks, uint64_t open, Copy copy)
        : copy_(copy), open_(open), done_(n_chunks) {
        pool_.reserve(want);   // (nothing is running yet: an exception of it goes to the caller)
        try {
            for (unsigned t = 0; t < want; ++t) pool_.emplace_back([this, t] { work(t); });
        } catch (...) {
        }
        count_.store((unsigned)pool_.size(), std::memory_order_release);
        started_.store(true, std::memory_order_release);
    }
    CopyThreads(const CopyThreads&) = delete;
    CopyThreads& operator=(const CopyThreads&) = delete;
    ~CopyThreads() {
        stop_.store(true);
        for (auto& t : pool_) t.join();
    }

    // Chunks below n may be filled.
    void open(uint64_t n) { open_.store(n, std::memory_order_release); }

    // Returns once chunk c, which has to be open, is copied.
    void wait(uint64_t c) {
        const unsigned T = count_.load(std::memory_order_relaxed);
        if (T == 0) copy_(c, 0, 1);
        while (done_[c].load(std::memory_order_acquire) < T) std::this_thread::yield();
    }

  private:
    void work(unsigned t) {
        while (!started_.load(std::memory_order_acquire)) std::this_thread::yield();
        const unsigned T = count_.load(std::memory_order_acquire);
        for (uint64_t c = 0; c < done_.size(); ++c) {
            while (open_.load(std::memory_order_acquire) <= c) {
                if (stop_.load(std::memory_order_relaxed)) return;
                std::this_thread::yield();
            }
            copy_(c, t, T);
            done_[c].fetch_add(1, std::memory_order_release);
        }
    }

    Copy copy_;
    std::atomic<unsigned> count_{0};
    std::atomic<bool> started_{false}, stop_{false};
    std::atomic<uint64_t> open_;
    std::vector<std::atomic<uint32_t>> done_;
    std::vector<std::thread> pool_;
};

}  // namespace cbh

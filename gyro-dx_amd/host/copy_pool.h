// Host copies between a caller's pageable memory and the engine's pinned staging slots, split over a few
// threads: one thread moves 8-10 GB/s (page faults of a fresh output included), a sixth of the host
// link. The helpers belong to one engine: they are started with its buffers where its calls can be
// large, sleep between calls and are joined with it.
#pragma once
#include <condition_variable>
#include <cstdint>
#include <cstring>
#include <deque>
#include <mutex>
#include <system_error>
#include <thread>
#include <vector>

namespace gyro {

class CopyPool {
  public:
    static constexpr uint64_t kPiece = 128u << 10;
    static constexpr uint64_t kParallelBytes = 1u << 20;  // a copy from here on is worth waking the helpers

    ~CopyPool() {
        {
            std::lock_guard<std::mutex> lock(mutex_);
            stop_ = true;
        }
        wake_.notify_all();
        for (std::thread &t : threads_) t.join();
    }

    // Starts the helpers, once (the first post does it at the latest); false where the system gives no thread.
    bool start() {
        if (!tried_) {
            tried_ = true;
            const unsigned cpus = std::thread::hardware_concurrency();
            const unsigned n = cpus > kHelpers ? kHelpers : (cpus > 1 ? cpus - 1 : 0);
            try {
                for (unsigned i = 0; i < n; ++i) threads_.emplace_back([this] { helper(); });
            } catch (const std::system_error &) {
            }
        }
        return !threads_.empty();
    }

    // Hands a copy to the helpers in pieces (or makes it at once where there are none); both ranges stay untouched by
    // the caller until finish() or drop(). Whole parts of a long download in place of pieces were no faster at any
    // size: 8 MB read back 0.25 against 0.23 ms, 32 MB into fresh pages 1.06 and 1.05, 48 MB 1.97 and 1.54.
    void post(void *dst, const void *src, uint64_t bytes) {
        if (!start()) {
            std::memcpy(dst, src, bytes);
            return;
        }
        {
            std::lock_guard<std::mutex> lock(mutex_);
            for (uint64_t at = 0; at < bytes; at += kPiece)
                queue_.push_back({static_cast<uint8_t *>(dst) + at, static_cast<const uint8_t *>(src) + at,
                                  bytes - at < kPiece ? bytes - at : kPiece});
        }
        if (bytes > kPiece) wake_.notify_all();
        else wake_.notify_one();
    }
    // Makes what is still queued beside the helpers and returns once every posted copy is complete.
    void finish() {
        std::unique_lock<std::mutex> lock(mutex_);
        run(lock);
        idle_.wait(lock, [this] { return running_ == 0; });
    }
    // Drops what is still queued and returns once no helper copies: nothing posted is touched after it.
    void drop() {
        std::unique_lock<std::mutex> lock(mutex_);
        queue_.clear();
        idle_.wait(lock, [this] { return running_ == 0; });
    }
    // Around posts whose ranges the caller may free once it is told of an error: however the block is left,
    // no copy is queued or running behind it.
    class Scope {
      public:
        explicit Scope(CopyPool &pool) : pool_(pool) {}
        ~Scope() { pool_.drop(); }
        Scope(const Scope &) = delete;
        Scope &operator=(const Scope &) = delete;

      private:
        CopyPool &pool_;
    };
    // memcpy, from kParallelBytes on in pieces over all threads.
    void copy(void *dst, const void *src, uint64_t bytes) {
        if (bytes < kParallelBytes) {
            std::memcpy(dst, src, bytes);
            return;
        }
        Scope scope(*this);
        post(dst, src, bytes);
        finish();
    }

  private:
    static constexpr unsigned kHelpers = 5;

    struct Piece {
        void *dst;
        const void *src;
        uint64_t bytes;
    };

    // Takes pieces until none is queued (the lock is held on entry and return, not while copying).
    void run(std::unique_lock<std::mutex> &lock) {
        while (!queue_.empty()) {
            const Piece p = queue_.front();
            queue_.pop_front();
            ++running_;
            lock.unlock();
            std::memcpy(p.dst, p.src, p.bytes);
            lock.lock();
            if (--running_ == 0 && queue_.empty()) idle_.notify_all();
        }
    }
    void helper() {
        std::unique_lock<std::mutex> lock(mutex_);
        for (;;) {
            wake_.wait(lock, [this] { return stop_ || !queue_.empty(); });
            if (stop_) return;
            run(lock);
        }
    }

    std::mutex mutex_;
    std::condition_variable wake_, idle_;
    std::deque<Piece> queue_;
    std::vector<std::thread> threads_;
    unsigned running_ = 0;
    bool stop_ = false, tried_ = false;
};

}  // namespace gyro

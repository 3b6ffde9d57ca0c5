// Host memory copied by a few threads: between a caller's memory and the pinned staging buffers of the host-to-host codec.
#pragma once
#include <atomic>
#include <condition_variable>
#include <cstddef>
#include <cstdint>
#include <cstring>
#include <mutex>
#include <system_error>
#include <thread>

namespace pmh {

constexpr int kCopyThreads = 4;  // measured: 26 / 38 / 41 / 41 GB/s with 1 / 2 / 4 / 8 copy threads

// The threads of one codec call, the caller's among them: made with its first copy, ended with the call.  (Made for each copy they
// cost 7 us apiece: of a round trip of 3 Mi elements through Q8_0, 1002 us, making them took 176 and the copies that were too short for
// them 152; it took 937 with these and no other change.)  Between two copies a helper looks for the next one for some 30 us, about as long as the caller takes to
// submit a chunk, and then sleeps.  Throws nothing: where a helper cannot be made, the others copy its share.
class CopyTeam {
    static constexpr size_t kMinPiece = (size_t)64 << 10;  // below twice this, waking a helper takes as long as the copy
    std::thread helpers_[kCopyThreads - 1];
    int made_ = 0;
    bool tried_ = false;
    std::mutex mutex_;
    std::condition_variable wake_;
    uint8_t *dst_ = nullptr;
    const uint8_t *src_ = nullptr;
    size_t bytes_ = 0, piece_ = 0;
    // The copy's number times 64 and the next piece of it, in one word: a helper that comes late to a copy takes nothing of the one behind it.
    std::atomic<uint64_t> next_{63};
    std::atomic<int> left_{0};  // pieces not copied yet
    std::atomic<bool> stop_{false};

    // Takes pieces of the present copy until none is left.
    void work() noexcept {
        uint64_t n = next_.load(std::memory_order_acquire);
        while ((n & 63) < kCopyThreads) {
            if (!next_.compare_exchange_weak(n, n + 1, std::memory_order_acq_rel, std::memory_order_acquire)) continue;
            const size_t off = piece_ * (size_t)(n & 63);  // (what describes a copy does not change before all of its pieces are copied)
            if (off < bytes_) memcpy(dst_ + off, src_ + off, bytes_ - off < piece_ ? bytes_ - off : piece_);
            left_.fetch_sub(1, std::memory_order_release);
            n = next_.load(std::memory_order_acquire);
        }
    }
    static void pause() noexcept {
#if defined(__x86_64__)
        __builtin_ia32_pause();
#endif
    }
    bool idle() const noexcept { return (next_.load(std::memory_order_acquire) & 63) >= kCopyThreads; }
    void serve() noexcept {
        while (true) {
            for (int i = 0; i < 1000 && idle() && !stop_.load(std::memory_order_acquire); i++) pause();
            if (idle() && !stop_.load(std::memory_order_acquire)) {
                std::unique_lock<std::mutex> lock(mutex_);
                wake_.wait(lock, [&] { return !idle() || stop_.load(std::memory_order_acquire); });
            }
            if (stop_.load(std::memory_order_acquire)) return;
            work();
        }
    }

public:
    CopyTeam() = default;
    CopyTeam(const CopyTeam &) = delete;
    CopyTeam &operator=(const CopyTeam &) = delete;
    ~CopyTeam() {
        {
            std::lock_guard<std::mutex> lock(mutex_);
            stop_.store(true, std::memory_order_release);
        }
        wake_.notify_all();
        for (int i = 0; i < made_; i++) helpers_[i].join();
    }
    void copy(void *dst, const void *src, size_t bytes) noexcept {
        if (bytes < 2 * kMinPiece) {
            memcpy(dst, src, bytes);
            return;
        }
        dst_ = (uint8_t *)dst, src_ = (const uint8_t *)src, bytes_ = bytes;
        piece_ = ((bytes + kCopyThreads - 1) / kCopyThreads + 4095) & ~(size_t)4095;  // (all of them together at least `bytes`)
        left_.store(kCopyThreads, std::memory_order_relaxed);
        {
            std::lock_guard<std::mutex> lock(mutex_);  // (a helper that is about to sleep sees the copy or is woken)
            next_.store((next_.load(std::memory_order_relaxed) | 63) + 1, std::memory_order_release);
        }
        if (made_ > 0) wake_.notify_all();
        if (!tried_) {
            tried_ = true;
            try {
                for (; made_ < kCopyThreads - 1; made_++) helpers_[made_] = std::thread([this] { serve(); });
            } catch (const std::exception &) {  // (as many as could be made)
            }
        }
        work();
        for (int i = 0; left_.load(std::memory_order_acquire) > 0; i++) {
            if (i < 1000) pause();
            else std::this_thread::yield();  // (fewer processors than threads)
        }
    }
};

}  // namespace pmh

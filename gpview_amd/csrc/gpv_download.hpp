// gpv_download.hpp -- results from the device into host memory.
//
// hipMemcpyAsync into pageable memory takes 15 to 25 us a call and then moves about
// 14 GB/s: it stages on one thread, after the copy.  Here kernels write into
// page-locked staging.  Small results go out in one launch and are copied on by the
// caller; larger ones in chunks, each copied on by the caller and up to kHelpers
// threads while the next ones arrive: 6 MB of states 430 -> 290 us, 8 MB of normals 640 ->
// 400, four small arrays 60 -> 15; six helpers were slower than three.  Staging and threads belong to a context (its
// lock is held by the caller) and go with it.
//
// Page-locked destinations need no staging: larger results are copied straight there, at
// 52 GB/s (222 MB of states 5.99 -> 4.23 ms, 10 MB 362 -> 248 us).  Small ones
// stay with the one launch (20 KB in four arrays: 25 us, 65 in four copies).
#pragma once

#include "gpv_internal.hpp"

#include <atomic>
#include <condition_variable>
#include <cstring>
#include <exception>
#include <mutex>
#include <thread>
#include <vector>

namespace gpv {

class Downloader {
public:
    struct Piece {
        void* dst;         // host
        const void* src;   // device
        size_t n;
    };

    ~Downloader() { close(); }

    // Copies the pieces (work queued on s before is included) and waits for them.
    hipError_t run(const Piece* p, int count, hipStream_t s)
    {
        size_t total = 0;
        for (int k = 0; k < count; ++k) total += up(p[k].n);
        if (total == 0) return hipStreamSynchronize(s);
        const bool one = total <= kSmall && count <= kCopyMax;
        hipError_t e = hipSuccess;
        total = 0;
        staged_.clear();
        for (int k = 0; k < count && e == hipSuccess; ++k) {
            if (!p[k].n) continue;
            if (direct(p[k].dst, one)) {
                e = hipMemcpyAsync(p[k].dst, p[k].src, p[k].n, hipMemcpyDeviceToHost, s);
            } else {
                staged_.push_back(p[k]);
                total += up(p[k].n);
            }
        }
        if (e == hipSuccess && total) {
            const int n = (int)staged_.size();
            if (open(one ? kSmall : kChunks * kChunkMax) == hipSuccess)
                return one ? small(staged_.data(), n, s) : large(staged_.data(), n, total, s);
            // no staging to be had: the runtime's own copies
            (void)hipGetLastError();
            for (int k = 0; k < n && e == hipSuccess; ++k)
                e = hipMemcpyAsync(staged_[k].dst, staged_[k].src, staged_[k].n, hipMemcpyDeviceToHost, s);
        }
        const hipError_t w = hipStreamSynchronize(s);
        return e == hipSuccess ? w : e;
    }

    void close()
    {
        {
            std::lock_guard<std::mutex> lk(mu_);
            quit_ = true;
        }
        cv_.notify_all();
        for (std::thread& t : threads_) t.join();
        threads_.clear();
        quit_ = false;
        started_ = false;
        for (hipEvent_t& e : ev_) {
            if (e) (void)hipEventDestroy(e);
            e = nullptr;
        }
        if (buf_) (void)hipHostFree(buf_);
        buf_ = nullptr;
        cap_ = 0;
    }

private:
    static constexpr size_t kAlign = 256;
    static constexpr size_t kSmall = size_t(256) << 10;   // one launch, no threads
    static constexpr int kChunks = 8;                     // of a round
    static constexpr size_t kChunkMin = size_t(512) << 10, kChunkMax = size_t(2) << 20;
    static constexpr int kHelpers = 3;
    static size_t up(size_t n) { return (n + kAlign - 1) / kAlign * kAlign; }

    // Whether the runtime copies to dst: to device memory always, to page-locked
    // memory where the results are not small.
    static bool direct(const void* dst, bool one)
    {
        hipPointerAttribute_t a{};
        if (hipPointerGetAttributes(&a, dst) != hipSuccess) {
            (void)hipGetLastError();   // pageable memory
            return false;
        }
        return a.type == hipMemoryTypeDevice || (!one && a.type != hipMemoryTypeUnregistered);
    }

    hipError_t open(size_t bytes)
    {
        if (bytes > cap_) {
            if (buf_) (void)hipHostFree(buf_);
            buf_ = nullptr;
            cap_ = 0;
            void* b = nullptr;
            const hipError_t e = hipHostMalloc(&b, bytes, hipHostMallocDefault);
            if (e != hipSuccess) return e;
            buf_ = static_cast<char*>(b);
            cap_ = bytes;
        }
        for (hipEvent_t& v : ev_) {
            if (v || bytes == kSmall) continue;
            const hipError_t e = hipEventCreateWithFlags(&v, hipEventDisableTiming);
            if (e != hipSuccess) {
                v = nullptr;
                return e;
            }
        }
        return hipSuccess;
    }

    hipError_t small(const Piece* p, int count, hipStream_t s)
    {
        CopyOut L{};
        size_t at = 0;
        int m = 0;
        for (int k = 0; k < count; ++k) {
            if (!p[k].n) continue;
            L.src[m] = static_cast<const char*>(p[k].src);
            L.dst[m] = buf_ + at;
            L.n[m++] = (int64_t)p[k].n;
            at += up(p[k].n);
        }
        launch_copy_out(L, m, s);
        hipError_t e = hipGetLastError();
        const hipError_t w = hipStreamSynchronize(s);
        if (e == hipSuccess) e = w;
        if (e != hipSuccess) return e;
        at = 0;
        for (int k = 0; k < count; ++k) {
            if (!p[k].n) continue;
            memcpy(p[k].dst, buf_ + at, p[k].n);
            at += up(p[k].n);
        }
        return hipSuccess;
    }

    hipError_t large(const Piece* p, int count, size_t total, hipStream_t s)
    {
        start();
        size_t chunk = (total / kChunks + kAlign) / kAlign * kAlign;
        chunk = chunk < kChunkMin ? kChunkMin : chunk > kChunkMax ? kChunkMax : chunk;
        int k = 0;
        size_t at = 0;   // within piece k
        while (k < count) {
            // a round: up to kChunks chunks, each from one piece
            {
                std::unique_lock<std::mutex> lk(mu_);
                cv_.wait(lk, [&] { return active_ == 0; });
                items_.clear();
                while (k < count && items_.size() < (size_t)kChunks) {
                    const size_t left = p[k].n - at, n = left < chunk ? left : chunk;
                    if (n) items_.push_back({static_cast<char*>(p[k].dst) + at, static_cast<const char*>(p[k].src) + at, n});
                    at += n;
                    if (at == p[k].n) {
                        ++k;
                        at = 0;
                    }
                }
                next_.store(0);
                ready_.store(0);
                done_.store(0);
                failed_.store(false);
                ++gen_;
            }
            const int n = (int)items_.size();
            if (!n) break;
            cv_.notify_all();
            hipError_t e = hipSuccess;
            int sent = 0;
            for (; sent < n && e == hipSuccess; ++sent) {
                CopyOut L{};
                L.src[0] = static_cast<const char*>(items_[sent].src);
                L.dst[0] = buf_ + (size_t)sent * kChunkMax;
                L.n[0] = (int64_t)items_[sent].n;
                launch_copy_out(L, 1, s);
                e = hipGetLastError();
                if (e == hipSuccess) e = hipEventRecord(ev_[sent], s);
            }
            for (int i = 0; i < n && e == hipSuccess; ++i) {
                e = hipEventSynchronize(ev_[i]);
                if (e == hipSuccess) ready_.store(i + 1, std::memory_order_release);
            }
            if (e != hipSuccess) {
                (void)hipStreamSynchronize(s);   // nothing writes the staging any more
                failed_.store(true);
                ready_.store(n, std::memory_order_release);
            }
            work();
            while (done_.load(std::memory_order_acquire) < n) std::this_thread::yield();
            if (e != hipSuccess) return e;
        }
        return hipSuccess;
    }

    // takes chunks until none is left
    void work()
    {
        const int n = (int)items_.size();
        for (;;) {
            const int i = next_.fetch_add(1);
            if (i >= n) return;
            for (int spin = 0; ready_.load(std::memory_order_acquire) <= i; ++spin)
                if (spin > 64) std::this_thread::yield();
            if (!failed_.load()) memcpy(items_[i].dst, buf_ + (size_t)i * kChunkMax, items_[i].n);
            done_.fetch_add(1, std::memory_order_release);
        }
    }

    void start()
    {
        if (started_) return;
        started_ = true;
        try {
            while ((int)threads_.size() < kHelpers) threads_.emplace_back([this] { helper(); });
        } catch (const std::exception&) {
            // the caller copies alone, or with those that started
        }
    }

    void helper()
    {
        uint64_t seen = 0;
        std::unique_lock<std::mutex> lk(mu_);
        for (;;) {
            cv_.wait(lk, [&] { return quit_ || gen_ != seen; });
            if (quit_) return;
            seen = gen_;
            ++active_;
            lk.unlock();
            work();
            lk.lock();
            if (--active_ == 0) cv_.notify_all();
        }
    }

    char* buf_ = nullptr;
    size_t cap_ = 0;
    hipEvent_t ev_[kChunks] = {};
    std::vector<std::thread> threads_;
    bool started_ = false;
    std::mutex mu_;
    std::condition_variable cv_;
    uint64_t gen_ = 0;      // of the round at hand (mu_)
    int active_ = 0;        // helpers in a round (mu_)
    bool quit_ = false;     // (mu_)
    std::vector<Piece> staged_;
    std::vector<Piece> items_;   // rewritten only while no helper is active
    std::atomic<int> next_{0}, ready_{0}, done_{0};
    std::atomic<bool> failed_{false};
};

}  // namespace gpv

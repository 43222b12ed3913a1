// mdx_transfer.h -- copies between the caller's pageable arrays and the device
// through a small ring of pinned memory (host code).
//
// A copy of pageable memory runs at 16 GB/s and faults the caller's fresh pages
// one by one; the link alone carries 55 GB/s into pinned memory. The data go
// chunk by chunk through the ring, and in a large transfer kWorkers threads that
// live for it move them between ring and caller beside the calling thread.
// Download of 1 M molecules (176 MB) 24.7 -> 6.2 ms, of 100 k 2.0 -> 0.7 ms.
#pragma once

#include <hip/hip_runtime.h>

#include <algorithm>
#include <condition_variable>
#include <cstring>
#include <deque>
#include <functional>
#include <mutex>
#include <system_error>
#include <thread>
#include <vector>

namespace mdx {

// A context's ring: up to kSlots chunks of kChunk bytes, as many as the context's
// largest transfer so far fills, made on first use and held while the context
// lives. 176 MB into fresh 4 KB pages with 8 threads: 9.7 ms with 8 x 2 MB, 12.0
// with 8 x 0.5 MB, 15 with 4 x 2 MB.
struct PinnedRing {
    static constexpr size_t kChunk = 2u << 20;
    static constexpr int kSlots = 8;
    static constexpr size_t kSmall = 256u << 10;
    char *mem = nullptr, *dev = nullptr;  // host and device address
    size_t size = 0;
    hipEvent_t ev[kSlots] = {};

    // Bytes held for transfers of at most `need` bytes in all: one slot of kSmall
    // bytes for the small states (16 MB and their events take 0.1 to 0.2 ms), else
    // no more chunks than the transfer has.
    static constexpr size_t bytes(size_t need) {
        if (need <= kSmall) return kSmall;
        const size_t chunks = need / kChunk + (need % kChunk != 0);
        return kChunk * (chunks < (size_t)kSlots ? chunks : (size_t)kSlots);
    }
    hipError_t open(size_t need) {
        need = bytes(need);
        if (mem && size >= need) return hipSuccess;
        if (mem) (void)hipHostFree(mem);
        mem = dev = nullptr;
        size = need;
        for (int k = 0; k < slots(); ++k)
            if (!ev[k]) {
                const hipError_t r = hipEventCreateWithFlags(&ev[k], hipEventDisableTiming);
                if (r != hipSuccess) return r;
            }
        void *p = nullptr;
        hipError_t r = hipHostMalloc(&p, need, 0);
        if (r != hipSuccess) return r;
        void *d = nullptr;
        r = hipHostGetDevicePointer(&d, p, 0);
        if (r != hipSuccess) {
            (void)hipHostFree(p);
            return r;
        }
        mem = (char *)p;
        dev = (char *)d;
        return hipSuccess;
    }
    int slots() const { return size > kSmall ? (int)(size / kChunk) : 1; }
    void close() {
        if (mem) (void)hipHostFree(mem);
        for (auto &e : ev)
            if (e) (void)hipEventDestroy(e);
        mem = dev = nullptr;
        for (auto &e : ev) e = nullptr;
    }
};

// One transfer: pieces of host memory that lie behind one another in a device
// range. The calling thread cuts chunks, works on jobs itself when no slot is
// free, and returns from finish() when every job is done.
struct HostPiece {
    char *host;
    size_t bytes;
};

class HostTransfer {
  public:
    // Two threads from 32 MB on. 150 k molecules (34 MB): 2.4 ms alone, 1.5 with
    // two, 0.9 with four; 1 M: 6.7 (15.8 into fresh memory), 6.2, 5.6. Below, one
    // thread is as fast (100 k molecules: 0.73 ms, 0.71 with two) and more of them
    // lose their CPUs to a caller's own spinning thread pool (a pass with a tensor
    // conversion behind it: 1.4 ms alone, 2.1 with two, 3.8 with four, 4.8 with
    // eight).
    static constexpr size_t kWorkers = 2, kManyBytes = 32u << 20;

    HostTransfer(PinnedRing &ring, hipStream_t stream, int device, size_t total,
                 size_t many = kManyBytes)
        : ring_(ring), stream_(stream) {
        const size_t want = ring.mem && total >= many ? kWorkers : 0;
        const unsigned hw = std::thread::hardware_concurrency();
        const size_t most = hw > 1 ? hw - 1 : 0;
        try {
            for (size_t k = 0; k < std::min(want, most); ++k)
                workers_.emplace_back([this, device] {
                    note(hipSetDevice(device));
                    work();
                });
        } catch (const std::system_error &) {
            // fewer threads, or none: the caller does the jobs
        }
    }
    ~HostTransfer() { (void)finish(); }
    HostTransfer(const HostTransfer &) = delete;
    HostTransfer &operator=(const HostTransfer &) = delete;

    // The device range [dev, dev + sum of the pieces) into the pieces, behind
    // what is on the stream.
    void to_host(const char *dev, const std::vector<HostPiece> &pieces) {
        if (!ring_.mem) return direct((char *)dev, pieces, hipMemcpyDeviceToHost);
        each_chunk(pieces, [&](size_t off, size_t len) {
            const int s = slot();
            note(hipMemcpyAsync(at(s), dev + off, len, hipMemcpyDeviceToHost, stream_));
            note(hipEventRecord(ring_.ev[s], stream_));
            push([this, s, off, len, pieces] {
                note(hipEventSynchronize(ring_.ev[s]));
                split(pieces, off, len, [&](char *host, size_t o, size_t n) {
                    memcpy(host, at(s) + o, n);
                });
                release(s);
            });
        });
    }
    // The pieces into the device range; the stream has the copies once wait()
    // returns.
    void to_device(char *dev, const std::vector<HostPiece> &pieces) {
        if (!ring_.mem) return direct(dev, pieces, hipMemcpyHostToDevice);
        each_chunk(pieces, [&](size_t off, size_t len) {
            const int s = slot();
            push([this, s, off, len, dev, pieces] {
                split(pieces, off, len, [&](char *host, size_t o, size_t n) {
                    memcpy(at(s) + o, host, n);
                });
                note(hipMemcpyAsync(dev + off, at(s), len, hipMemcpyHostToDevice, stream_));
                note(hipEventRecord(ring_.ev[s], stream_));
                note(hipEventSynchronize(ring_.ev[s]));  // the slot is free again
                release(s);
            });
        });
    }
    void host_copy(void *dst, const void *src, size_t bytes) {
        for (size_t o = 0; o < bytes; o += PinnedRing::kChunk) {
            const size_t n = std::min(PinnedRing::kChunk, bytes - o);
            push([dst, src, o, n] { memcpy((char *)dst + o, (const char *)src + o, n); });
        }
    }
    // All jobs done.
    void wait() {
        while (run_one()) {
        }
        std::unique_lock<std::mutex> l(mu_);
        idle_cv_.wait(l, [this] { return jobs_.empty() && active_ == 0; });
    }
    hipError_t finish() {
        wait();
        {
            std::lock_guard<std::mutex> l(mu_);
            closed_ = true;
        }
        job_cv_.notify_all();
        for (auto &t : workers_) t.join();
        workers_.clear();
        return err_;
    }

  private:
    // without a ring (no pinned memory left): pageable copies
    void direct(char *dev, const std::vector<HostPiece> &pieces, hipMemcpyKind kind) {
        for (const HostPiece &p : pieces) {
            char *dst = kind == hipMemcpyDeviceToHost ? p.host : dev;
            char *src = kind == hipMemcpyDeviceToHost ? dev : p.host;
            note(hipMemcpyAsync(dst, src, p.bytes, kind, stream_));
            dev += p.bytes;
        }
        note(hipStreamSynchronize(stream_));
    }
    char *at(int s) { return ring_.mem + (size_t)s * PinnedRing::kChunk; }
    void note(hipError_t e) {
        if (e == hipSuccess) return;
        std::lock_guard<std::mutex> l(mu_);
        if (err_ == hipSuccess) err_ = e;
    }
    template <typename F> void each_chunk(const std::vector<HostPiece> &pieces, F f) {
        size_t total = 0;
        for (const HostPiece &p : pieces) total += p.bytes;
        for (size_t o = 0; o < total; o += PinnedRing::kChunk)
            f(o, std::min(PinnedRing::kChunk, total - o));
    }
    // f(host, offset in the chunk, bytes) for the parts of pieces in [off, off + len)
    template <typename F>
    static void split(const std::vector<HostPiece> &pieces, size_t off, size_t len, F f) {
        size_t p0 = 0;
        for (const HostPiece &p : pieces) {
            const size_t a = std::max(off, p0), b = std::min(off + len, p0 + p.bytes);
            if (a < b) f(p.host + (a - p0), a - off, b - a);
            p0 += p.bytes;
        }
    }
    int slot() {
        for (;;) {
            {
                std::unique_lock<std::mutex> l(mu_);
                for (int s = 0; s < ring_.slots(); ++s)
                    if (!busy_[s]) {
                        busy_[s] = true;
                        return s;
                    }
                if (jobs_.empty()) {  // a worker holds each slot and will free it
                    slot_cv_.wait(l);
                    continue;
                }
            }
            (void)run_one();
        }
    }
    void release(int s) {
        {
            std::lock_guard<std::mutex> l(mu_);
            busy_[s] = false;
        }
        slot_cv_.notify_one();
    }
    void push(std::function<void()> job) {
        {
            std::lock_guard<std::mutex> l(mu_);
            jobs_.push_back(std::move(job));
        }
        job_cv_.notify_one();
    }
    std::function<void()> take() {
        std::function<void()> job = std::move(jobs_.front());
        jobs_.pop_front();
        ++active_;
        return job;
    }
    void done() {
        std::lock_guard<std::mutex> l(mu_);
        if (--active_ == 0 && jobs_.empty()) idle_cv_.notify_all();
    }
    bool run_one() {
        std::function<void()> job;
        {
            std::lock_guard<std::mutex> l(mu_);
            if (jobs_.empty()) return false;
            job = take();
        }
        job();
        done();
        return true;
    }
    void work() {
        for (;;) {
            std::function<void()> job;
            {
                std::unique_lock<std::mutex> l(mu_);
                job_cv_.wait(l, [this] { return closed_ || !jobs_.empty(); });
                if (jobs_.empty()) return;
                job = take();
            }
            job();
            done();
        }
    }

    PinnedRing &ring_;
    hipStream_t stream_;
    std::vector<std::thread> workers_;
    std::mutex mu_;
    std::condition_variable job_cv_, slot_cv_, idle_cv_;
    std::deque<std::function<void()>> jobs_;
    bool busy_[PinnedRing::kSlots] = {};
    int active_ = 0;
    bool closed_ = false;
    hipError_t err_ = hipSuccess;
};

}  // namespace mdx

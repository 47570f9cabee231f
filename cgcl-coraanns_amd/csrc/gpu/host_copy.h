// Large host arrays to the device and back for the index-build tools, whose callers hold
// ordinary (pageable) arrays.
//
// The runtime copies a pageable array to the device at 36 GB/s (28 from 64 MiB) and back at
// 17 GB/s while the caller waits; a DMA from page-locked memory runs at 57 GB/s. Here a few
// host threads copy 4 MiB pieces into page-locked buffers (one thread copies 10-15 GB/s) and
// queue their DMAs on a stream of their own, and the caller's kernels for a chunk of rows are
// launched as soon as the chunk is queued, so that they run while the following chunks travel.
//
// A staging set (threads, their page-locked buffers, a stream, events) belongs to one call
// from its first large copy to its end; at most kKeepSets a device are kept for later calls, so
// calls from several host threads never share one. The threads of a set sleep between copies,
// and sleep while they wait for a buffer's DMA (hipEventBlockingSync): with threads started by
// each copy, and waits that spun, repeated calls took one or two scheduler ticks of 4 ms longer
// now and then (assign 12 MB 0.75 or 4.0 ms; the copy alone shows none of it).
#pragma once

#include <hip/hip_runtime.h>
#include <string.h>

#include <algorithm>
#include <atomic>
#include <condition_variable>
#include <mutex>
#include <new>
#include <system_error>
#include <thread>
#include <vector>

namespace cora {

constexpr size_t kPieceBytes = size_t{4} << 20;
constexpr int kCopyThreads = 4;  // 3, 4 and 6 copy alike
constexpr int kKeepSets = 2;
// Below these the runtime's copy is as fast. Up: plain 0.24 / 0.46 / 0.94 / 1.43 / 2.58 ms for 8, 16,
// 32, 40 and 64 MiB, staged 0.27 / 0.46 / 0.82 / 1.01 / 1.58 (a whole assign of 32 MiB: 1.25 and
// 1.40 ms, of 64 MiB 2.77 and 2.41). Down: plain 0.25 / 0.49 / 0.98 / 2.03 for 4, 8, 16 and 32 MiB,
// staged 0.30 / 0.38 / 0.58 / 0.99.
constexpr size_t kStagedUpBytes = size_t{40} << 20;
constexpr size_t kStagedDownBytes = size_t{8} << 20;

struct StagingSet {
    int device = 0;
    StagingSet *next = nullptr;  // in the pool
    hipStream_t stream = nullptr;
    hipEvent_t mark = nullptr;
    void *buf[2 * kCopyThreads] = {};
    hipEvent_t ev[2 * kCopyThreads] = {};

    bool create(int dev) {
        device = dev;
        if (hipStreamCreateWithFlags(&stream, hipStreamNonBlocking) != hipSuccess ||
            hipEventCreateWithFlags(&mark, hipEventDisableTiming) != hipSuccess)
            return false;
        for (int i = 0; i < 2 * kCopyThreads; ++i)
            if (hipHostMalloc(&buf[i], kPieceBytes, hipHostMallocDefault) != hipSuccess ||
                hipEventCreateWithFlags(&ev[i], hipEventDisableTiming | hipEventBlockingSync) != hipSuccess)
                return false;
        for (; threads_ < kCopyThreads; ++threads_) {
            try {
                thread_[threads_] = std::thread([this, t = threads_] { serve(t); });
            } catch (const std::system_error &) {
                break;
            }
        }
        return threads_ > 0;
    }
    ~StagingSet() {
        {
            std::lock_guard<std::mutex> lock(mu_);
            quit_ = true;
        }
        wake_.notify_all();
        for (int t = 0; t < threads_; ++t)
            thread_[t].join();
        for (int i = 0; i < 2 * kCopyThreads; ++i) {
            if (ev[i])
                (void)hipEventDestroy(ev[i]);
            if (buf[i])
                (void)hipHostFree(buf[i]);
        }
        if (mark)
            (void)hipEventDestroy(mark);
        if (stream)
            (void)hipStreamDestroy(stream);
    }

    // work(t) on the threads t = 0 .. min(pieces, threads) - 1; join() ends the job. work lives
    // until then and throws nothing.
    template <class W>
    void start(W &work, size_t pieces) {
        std::lock_guard<std::mutex> lock(mu_);
        arg_ = &work;
        fn_ = [](void *w, int t) { (*static_cast<W *>(w))(t); };
        want_ = active_ = (int)std::min<size_t>(threads_, pieces);
        ++job_;
        wake_.notify_all();
    }
    void join() {
        std::unique_lock<std::mutex> lock(mu_);
        done_.wait(lock, [&] { return active_ == 0; });
    }

  private:
    void serve(int t) {
        uint64_t seen = 0;
        std::unique_lock<std::mutex> lock(mu_);
        for (;;) {
            wake_.wait(lock, [&] { return quit_ || job_ != seen; });
            if (quit_)
                return;
            seen = job_;
            if (t >= want_)
                continue;
            lock.unlock();
            fn_(arg_, t);
            lock.lock();
            if (--active_ == 0)
                done_.notify_all();
        }
    }

    std::mutex mu_;
    std::condition_variable wake_, done_;
    uint64_t job_ = 0;
    int want_ = 0, active_ = 0, threads_ = 0;
    bool quit_ = false;
    void *arg_ = nullptr;
    void (*fn_)(void *, int) = nullptr;
    std::thread thread_[kCopyThreads];
};

// The idle sets. Never destroyed: at the process's end the runtime may already be gone (the
// sets' threads sleep until then).
struct StagingPool {
    std::mutex mu;
    StagingSet *idle = nullptr;
    StagingSet *take(int device) {
        std::lock_guard<std::mutex> lock(mu);
        for (StagingSet **p = &idle; *p; p = &(*p)->next)
            if ((*p)->device == device) {
                StagingSet *s = *p;
                *p = s->next;
                return s;
            }
        return nullptr;
    }
    bool keep(StagingSet *s) {
        std::lock_guard<std::mutex> lock(mu);
        int n = 0;
        for (StagingSet *i = idle; i; i = i->next)
            n += i->device == s->device;
        if (n >= kKeepSets)
            return false;
        s->next = idle;
        idle = s;
        return true;
    }
};
inline StagingPool &staging_pool() {
    static StagingPool *pool = new StagingPool();
    return *pool;
}

// A staging set of the current device from the first large copy to the end of this object (none:
// plain copies). A call of small arrays takes none: making one costs far more than its copies.
class Staging {
  public:
    explicit Staging(int device) : device_(device) {}
    ~Staging() {
        if (!set_)
            return;
        // nothing of this call may still use the buffers
        (void)hipStreamSynchronize(set_->stream);
        if (!staging_pool().keep(set_))
            delete set_;
    }
    Staging(const Staging &) = delete;
    Staging &operator=(const Staging &) = delete;

    // src [bytes] to dst, in chunks of chunk_bytes; for each chunk in turn, once the null stream is
    // ordered behind its copy, launch(offset, length) queues the work that reads it (0, or an
    // error that ends the call). The host array may be reused when this returns; the device
    // work is still in flight.
    template <class F>
    hipError_t upload(const void *src, void *dst, size_t bytes, size_t chunk_bytes, int &rc, F launch) {
        rc = 0;
        const size_t nchunks = (bytes + chunk_bytes - 1) / chunk_bytes;
        if (bytes >= kStagedUpBytes && acquire()) {
            std::vector<uint32_t> left;  // pieces of each chunk that are not queued yet
            bool room = true;
            try {
                left.resize(nchunks);
            } catch (const std::bad_alloc &) {
                room = false;
            }
            if (room)
                return staged_upload(src, dst, bytes, chunk_bytes, left, rc, launch);
        }
        for (size_t c = 0; c < nchunks; ++c) {
            const size_t o = c * chunk_bytes, len = std::min(chunk_bytes, bytes - o);
            const hipError_t r = hipMemcpy(static_cast<char *>(dst) + o, static_cast<const char *>(src) + o, len,
                                           hipMemcpyHostToDevice);
            if (r != hipSuccess)
                return r;
            if ((rc = launch(o, len)) != 0)
                return hipSuccess;
        }
        return hipSuccess;
    }

    // src (device, written by work already on the null stream) to dst [bytes]; complete on return.
    hipError_t download(const void *src, void *dst, size_t bytes) {
        if (bytes >= kStagedDownBytes && acquire())
            return staged_download(src, dst, bytes);
        return hipMemcpy(dst, src, bytes, hipMemcpyDeviceToHost);
    }

  private:
    bool acquire() {
        if (set_ || tried_)
            return set_ != nullptr;
        tried_ = true;
        set_ = staging_pool().take(device_);
        if (set_)
            return true;
        set_ = new (std::nothrow) StagingSet();
        if (set_ && !set_->create(device_)) {
            (void)hipGetLastError();
            delete set_;
            set_ = nullptr;
        }
        return set_ != nullptr;
    }

    template <class F>
    hipError_t staged_upload(const void *src, void *dst, size_t bytes, size_t chunk_bytes, std::vector<uint32_t> &left,
                             int &rc, F &launch) {
        const size_t nchunks = left.size();
        const size_t per = (chunk_bytes + kPieceBytes - 1) / kPieceBytes;  // pieces of a whole chunk
        size_t pieces = 0;
        for (size_t c = 0; c < nchunks; ++c) {
            left[c] = (uint32_t)((std::min(chunk_bytes, bytes - c * chunk_bytes) + kPieceBytes - 1) / kPieceBytes);
            pieces += left[c];
        }
        std::mutex mu;
        std::condition_variable cv;
        std::atomic<size_t> next{0};
        std::atomic<bool> stop{false};
        hipError_t worker_err = hipSuccess;
        auto work = [&](int t) {
            hipError_t e = hipSetDevice(set_->device);
            for (int b = 0; e == hipSuccess && !stop.load(); b ^= 1) {
                const size_t i = next.fetch_add(1);
                if (i >= pieces)
                    return;
                const size_t c = i / per, off = c * chunk_bytes + i % per * kPieceBytes;
                const size_t len = std::min({kPieceBytes, (c + 1) * chunk_bytes - off, bytes - off});
                const int slot = 2 * t + b;
                e = hipEventSynchronize(set_->ev[slot]);  // the buffer's last copy (none: at once)
                if (e != hipSuccess)
                    break;
                memcpy(set_->buf[slot], static_cast<const char *>(src) + off, len);
                std::lock_guard<std::mutex> lock(mu);
                e = hipMemcpyAsync(static_cast<char *>(dst) + off, set_->buf[slot], len, hipMemcpyHostToDevice,
                                   set_->stream);
                if (e == hipSuccess)
                    e = hipEventRecord(set_->ev[slot], set_->stream);
                if (e == hipSuccess && --left[c] == 0)
                    cv.notify_all();
            }
            if (e != hipSuccess) {
                std::lock_guard<std::mutex> lock(mu);
                worker_err = e;
                stop = true;
                cv.notify_all();
            }
        };
        set_->start(work, pieces);
        hipError_t err = hipSuccess;
        for (size_t c = 0; c < nchunks && err == hipSuccess && rc == 0; ++c) {
            {
                std::unique_lock<std::mutex> lock(mu);
                cv.wait(lock, [&] { return left[c] == 0 || worker_err != hipSuccess; });
                err = worker_err;
            }
            // (the marker may lie behind pieces of later chunks: a little late, never early)
            if (err == hipSuccess)
                err = hipEventRecord(set_->mark, set_->stream);
            if (err == hipSuccess)
                err = hipStreamWaitEvent(nullptr, set_->mark, 0);
            if (err == hipSuccess)
                rc = launch(c * chunk_bytes, std::min(chunk_bytes, bytes - c * chunk_bytes));
        }
        if (err != hipSuccess || rc != 0)
            stop = true;
        set_->join();
        return err;
    }

    hipError_t staged_download(const void *src, void *dst, size_t bytes) {
        const size_t pieces = (bytes + kPieceBytes - 1) / kPieceBytes;
        hipError_t err = hipEventRecord(set_->mark, nullptr);
        if (err == hipSuccess)
            err = hipStreamWaitEvent(set_->stream, set_->mark, 0);
        if (err != hipSuccess)
            return err;
        std::mutex mu;
        std::atomic<size_t> next{0};
        std::atomic<bool> stop{false};
        hipError_t worker_err = hipSuccess;
        auto work = [&](int t) {
            hipError_t e = hipSetDevice(set_->device);
            // two pieces in turn: one on its way while the other is copied out
            size_t at[2], len[2] = {0, 0};
            const auto out = [&](int b) {
                if (!len[b])
                    return;
                if (e == hipSuccess)
                    e = hipEventSynchronize(set_->ev[2 * t + b]);
                if (e == hipSuccess)
                    memcpy(static_cast<char *>(dst) + at[b], set_->buf[2 * t + b], len[b]);
                len[b] = 0;
            };
            int b = 0;
            for (; e == hipSuccess && !stop.load(); b ^= 1) {
                out(b);
                const size_t i = next.fetch_add(1);
                if (i >= pieces || e != hipSuccess)
                    break;
                at[b] = i * kPieceBytes;
                const size_t l = std::min(kPieceBytes, bytes - at[b]);
                std::lock_guard<std::mutex> lock(mu);
                e = hipMemcpyAsync(set_->buf[2 * t + b], static_cast<const char *>(src) + at[b], l,
                                   hipMemcpyDeviceToHost, set_->stream);
                if (e == hipSuccess)
                    e = hipEventRecord(set_->ev[2 * t + b], set_->stream);
                if (e == hipSuccess)
                    len[b] = l;
            }
            out(b);
            out(b ^ 1);
            if (e != hipSuccess) {
                std::lock_guard<std::mutex> lock(mu);
                worker_err = e;
                stop = true;
            }
        };
        set_->start(work, pieces);
        set_->join();
        return worker_err;
    }

    int device_;
    bool tried_ = false;
    StagingSet *set_ = nullptr;
};

}  // namespace cora

// Staging of downloads and uploads, shared by a device's contexts.
#pragma once
#include <hip/hip_runtime.h>

#include <algorithm>
#include <atomic>
#include <condition_variable>
#include <cstddef>
#include <mutex>
#include <thread>
#include <vector>

namespace mfs {

// A field crosses in chunks: a kernel reorders a chunk on the device, one
// copy moves it between a device slot and a pinned host slot, and a host
// thread copies between the slot and the caller's array, which is pageable and
// often not yet backed by memory (its page faults are most of a large
// download's host time).  Several threads work chunks at once, each with a
// slot, so that the reorder, the link and the host's copies overlap.  Before,
// one host thread scattered the whole field out of a pageable copy of its
// device array: the five state fields of 6.0M cells took 340 ms and the three
// gradients 238.  Now they take 10 and 22 ms, and uploading the five state
// fields 10 instead of 430 (in part the reads and writes of whole state
// buffers per field).
constexpr int kIoSlots = 8;
constexpr size_t kIoValues = (size_t)1 << 18;  // values per chunk (2 MiB)
struct IoSlot {
    double *host = nullptr, *dev = nullptr;
    hipEvent_t done = nullptr;
    bool taken = false;
};

// The slots of a device: allocated as chunks need them and freed with the
// device's last context.  A thread holds one for a chunk at a time, so the
// transfers of several contexts share them, and no lock is held meanwhile.
class IoPool {
  public:
    void join() {
        std::lock_guard<std::mutex> lk(mu_);
        ++users_;
    }
    void leave() {
        std::lock_guard<std::mutex> lk(mu_);
        if (--users_ > 0) return;
        for (IoSlot& s : slot_) {
            if (s.host) (void)hipHostFree(s.host);
            if (s.dev) (void)hipFree(s.dev);
            if (s.done) (void)hipEventDestroy(s.done);
            s = IoSlot{};
        }
    }
    // Moves `count` values of a context on `device`, chunk by chunk:
    // move(slot, first value, values) enqueues a chunk's work on `stream`, up
    // to the record of the slot's event, and finish(slot, first, values) does
    // its host part after the event.  Returns the first error.
    template <typename Move, typename Finish>
    hipError_t transfer(int device, hipStream_t stream, size_t count, Move&& move, Finish&& finish) {
        const size_t chunks = (count + kIoValues - 1) / kIoValues;
        std::atomic<size_t> next{0};
        std::atomic<int> failed{(int)hipSuccess};
        auto work = [&] {
            hipError_t e = hipSetDevice(device);
            while (e == hipSuccess && failed.load() == (int)hipSuccess) {
                const size_t c = next.fetch_add(1);
                if (c >= chunks) return;
                IoSlot& s = take();
                e = complete(s);
                const size_t t0 = c * kIoValues, n = std::min(kIoValues, count - t0);
                if (e == hipSuccess) e = move(s, t0, n);
                if (e == hipSuccess) e = hipEventSynchronize(s.done);
                if (e == hipSuccess)
                    finish(s, t0, n);
                else
                    (void)hipStreamSynchronize(stream);  // nothing enqueued touches the slot any more
                put(s);
            }
            int none = (int)hipSuccess;
            if (e != hipSuccess) failed.compare_exchange_strong(none, (int)e);
        };
        const int threads =
            (int)std::min<size_t>({(size_t)kIoSlots, chunks, std::max<size_t>(1, std::thread::hardware_concurrency())});
        std::vector<std::thread> th;
        try {
            th.reserve(threads);
            for (int k = 1; k < threads; ++k) th.emplace_back(work);
        } catch (...) {  // fewer helpers: the calling thread takes every chunk that is left
        }
        work();
        for (auto& t : th) t.join();
        return (hipError_t)failed.load();
    }

  private:
    // A free slot, one that has its memory first.
    IoSlot& take() {
        std::unique_lock<std::mutex> lk(mu_);
        while (true) {
            IoSlot* best = nullptr;
            for (IoSlot& s : slot_)
                if (!s.taken && (!best || (s.done && !best->done))) best = &s;
            if (best) {
                best->taken = true;
                return *best;
            }
            freed_.wait(lk);
        }
    }
    void put(IoSlot& s) {
        {
            std::lock_guard<std::mutex> lk(mu_);
            s.taken = false;
        }
        freed_.notify_one();
    }
    hipError_t complete(IoSlot& s) {
        hipError_t e = hipSuccess;
        if (!s.host) e = hipHostMalloc((void**)&s.host, kIoValues * sizeof(double), 0);
        if (e == hipSuccess && !s.dev) e = hipMalloc((void**)&s.dev, kIoValues * sizeof(double));
        if (e == hipSuccess && !s.done) e = hipEventCreateWithFlags(&s.done, hipEventDisableTiming);
        return e;
    }

    std::mutex mu_;
    std::condition_variable freed_;
    int users_ = 0;
    IoSlot slot_[kIoSlots];
};

}  // namespace mfs

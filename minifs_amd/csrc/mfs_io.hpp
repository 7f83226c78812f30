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
    hipEvent_t done = nullptr;  // set: the slot has its memory
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
        for (IoSlot& s : slot_) strip(s);
    }
    // Moves `count` values of a context on `device`, chunk by chunk:
    // move(slot, first value, values) enqueues a chunk's work on `stream` and
    // finish(slot, first, values) does its host part after it.  Returns the
    // first error.  Where there is no memory for further slots the threads
    // share those there are; without any the calling thread goes through
    // `spare`, device memory of spare_values values that the context has idle,
    // and pageable memory.
    template <typename Move, typename Finish>
    hipError_t transfer(int device, hipStream_t stream, size_t count, double* spare, size_t spare_values, Move&& move,
                        Finish&& finish) {
        const size_t chunks = (count + kIoValues - 1) / kIoValues;
        std::atomic<size_t> next{0};
        std::atomic<int> failed{(int)hipSuccess};
        std::atomic<bool> more{true}, none{false};  // memory for further slots; no slot at all
        auto work = [&] {
            hipError_t e = hipSetDevice(device);
            while (e == hipSuccess && failed.load() == (int)hipSuccess && !none) {
                const size_t c = next.fetch_add(1);
                if (c >= chunks) return;
                IoSlot* s = take(more);
                if (s && !complete(*s)) {
                    more = false;
                    put(*s);
                    s = take(false);
                }
                if (!s) {
                    none = true;
                    return;
                }
                const size_t t0 = c * kIoValues, n = std::min(kIoValues, count - t0);
                e = move(*s, t0, n);
                if (e == hipSuccess) e = hipEventRecord(s->done, stream);
                if (e == hipSuccess) e = hipEventSynchronize(s->done);
                if (e == hipSuccess)
                    finish(*s, t0, n);
                else
                    (void)hipStreamSynchronize(stream);  // nothing enqueued touches the slot any more
                put(*s);
            }
            int unset = (int)hipSuccess;
            if (e != hipSuccess) failed.compare_exchange_strong(unset, (int)e);
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
        hipError_t e = (hipError_t)failed.load();
        if (!none || e != hipSuccess) return e;
        std::lock_guard<std::mutex> lk(spare_mu_);  // two transfers of one context share its spare memory
        std::vector<double> host;
        try {
            host.resize(std::min(count, spare_values));
        } catch (...) {
            return hipErrorOutOfMemory;
        }
        IoSlot s;
        s.host = host.data();
        s.dev = spare;
        for (size_t t0 = 0; t0 < count && e == hipSuccess; t0 += host.size()) {
            const size_t n = std::min(host.size(), count - t0);
            e = move(s, t0, n);
            const hipError_t w = hipStreamSynchronize(stream);
            if (e == hipSuccess) e = w;
            if (e == hipSuccess) finish(s, t0, n);
        }
        return e;
    }

  private:
    // A free slot, one that has its memory first; with `more` one that has
    // none yet, otherwise null where no slot has any.
    IoSlot* take(bool more) {
        std::unique_lock<std::mutex> lk(mu_);
        while (true) {
            IoSlot* best = nullptr;
            bool busy = false;
            for (IoSlot& s : slot_) {
                busy = busy || s.taken;
                if (!s.taken && (s.done || more) && (!best || (s.done && !best->done))) best = &s;
            }
            if (best) {
                best->taken = true;
                return best;
            }
            if (!busy) return nullptr;
            freed_.wait(lk);
        }
    }
    void put(IoSlot& s) {
        {
            std::lock_guard<std::mutex> lk(mu_);
            s.taken = false;
        }
        freed_.notify_all();
    }
    // Gives a taken slot its memory, all or none of it.
    static bool complete(IoSlot& s) {
        if (s.done) return true;
        const size_t bytes = kIoValues * sizeof(double);
        if (hipHostMalloc((void**)&s.host, bytes, 0) == hipSuccess && hipMalloc((void**)&s.dev, bytes) == hipSuccess &&
            hipEventCreateWithFlags(&s.done, hipEventDisableTiming) == hipSuccess)
            return true;
        strip(s);
        (void)hipGetLastError();  // a launch check that follows must not find it
        return false;
    }
    static void strip(IoSlot& s) {
        if (s.host) (void)hipHostFree(s.host);
        if (s.dev) (void)hipFree(s.dev);
        if (s.done) (void)hipEventDestroy(s.done);
        s.host = s.dev = nullptr;
        s.done = nullptr;
    }

    std::mutex mu_, spare_mu_;
    std::condition_variable freed_;
    int users_ = 0;
    IoSlot slot_[kIoSlots];
};

}  // namespace mfs

// The staging slots of downloads and uploads (minifs_amd/csrc/mfs_io.hpp) on
// a runtime of its own, in host memory.  Built and run by test_io_pool.py:
//   io_pool scenario
// prints "ok", or what is wrong.
#include <chrono>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <future>
#include <string>

#include "mfs_io.hpp"

namespace {
std::mutex mu;
int room = 1000, held = 0, most = 0, syncs = 0;  // allocations that succeed, held, most held; stream waits
thread_local hipError_t last_error = hipSuccess;
hipError_t allocate(void** p, size_t bytes) {
    std::lock_guard<std::mutex> lk(mu);
    if (held >= room) return last_error = hipErrorOutOfMemory;
    most = std::max(most, ++held);
    *p = std::malloc(bytes);
    return hipSuccess;
}
hipError_t release(void* p) {
    std::lock_guard<std::mutex> lk(mu);
    --held;
    std::free(p);
    return hipSuccess;
}
}  // namespace

extern "C" {
hipError_t hipMalloc(void** p, size_t bytes) { return allocate(p, bytes); }
hipError_t hipHostMalloc(void** p, size_t bytes, unsigned) { return allocate(p, bytes); }
hipError_t hipFree(void* p) { return release(p); }
hipError_t hipHostFree(void* p) { return release(p); }
hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) {
    *e = reinterpret_cast<hipEvent_t>(new char);
    return hipSuccess;
}
hipError_t hipEventDestroy(hipEvent_t e) {
    delete reinterpret_cast<char*>(e);
    return hipSuccess;
}
hipError_t hipEventRecord(hipEvent_t e, hipStream_t) { return e ? hipSuccess : hipErrorInvalidHandle; }
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) {
    std::lock_guard<std::mutex> lk(mu);
    ++syncs;
    return hipSuccess;
}
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipGetLastError() {
    const hipError_t e = last_error;
    last_error = hipSuccess;
    return e;
}
}

namespace {
using mfs::IoSlot;

// A download of `count` values k -> base + k; hold() runs in every chunk.
template <typename Hold>
std::string download(mfs::IoPool& pool, size_t count, double base, Hold&& hold) {
    std::vector<double> out(count, -1.0), spare(777);
    const hipError_t e = pool.transfer(
        0, nullptr, count, spare.data(), spare.size(),
        [&](IoSlot& s, size_t t0, size_t n) {
            for (size_t k = 0; k < n; ++k) s.dev[k] = base + (double)(t0 + k);
            std::memcpy(s.host, s.dev, n * sizeof(double));
            return hipGetLastError();
        },
        [&](IoSlot& s, size_t t0, size_t n) {
            hold();
            std::memcpy(out.data() + t0, s.host, n * sizeof(double));
        });
    if (e != hipSuccess) return "error " + std::to_string((int)e);
    for (size_t k = 0; k < count; ++k)
        if (out[k] != base + (double)k) return "wrong value " + std::to_string(k);
    return "";
}
const auto nothing = [] {};

std::string run(const std::string& what) {
    const size_t V = mfs::kIoValues;
    mfs::IoPool pool;
    pool.join();
    std::string e;
    if (what == "sizes")
        for (size_t n : {(size_t)0, (size_t)1, V - 1, V, V + 1, 7 * V, 40 * V + 3}) {
            e = e.empty() ? download(pool, n, (double)n, nothing) : e;
            if (most > 2 * mfs::kIoSlots) e = "more than the slots";
        }
    if (what == "two contexts") {
        // another context is created, downloads and is destroyed while a
        // download is held up in one of its chunks
        std::promise<void> inside, done;
        std::atomic<bool> first{true};
        std::string e1;
        std::thread one([&] {
            e1 = download(pool, 5 * V, 1.0, [&] {
                if (!first.exchange(false)) return;
                inside.set_value();
                if (done.get_future().wait_for(std::chrono::seconds(20)) != std::future_status::ready)
                    e = "the second context waited for the first one's download";
            });
        });
        inside.get_future().wait();
        pool.join();
        const std::string e2 = download(pool, 30 * V, 2.0, nothing);
        pool.leave();
        done.set_value();
        one.join();
        if (e.empty()) e = e1 + e2;
    }
    if (what == "many at once") {
        std::vector<std::string> es(12);
        std::vector<std::thread> th;
        for (int k = 0; k < 12; ++k) th.emplace_back([&, k] { es[k] = download(pool, (k + 1) * V + k, k, nothing); });
        for (auto& t : th) t.join();
        for (auto& x : es) e += x;
        if (most > 2 * mfs::kIoSlots) e = "more than the slots";
    }
    if (what == "failed chunk") {
        std::atomic<int> calls{0};
        const hipError_t r = pool.transfer(
            0, nullptr, 20 * V, nullptr, 0, [&](IoSlot&, size_t, size_t) { return ++calls == 3 ? hipErrorUnknown : hipSuccess; },
            [](IoSlot&, size_t, size_t) {});
        if (r != hipErrorUnknown) e = "the error is lost";
        if (syncs == 0) e = "a slot is given back before its chunk's work has ended";
        if (e.empty()) e = download(pool, 20 * V, 3.0, nothing);  // every slot is free again
    }
    if (what == "no memory")  // for no slot, half of one, one, one and a half, three
        for (int r : {0, 1, 2, 3, 6}) {
            room = r;
            if (e.empty()) e = download(pool, 20 * V + 5, r, nothing);
            if (e.empty()) e = download(pool, 3, r, nothing);
            if (e.empty() && held > r - r % 2) e = "half a slot is kept";
        }
    if (what == "no memory, many at once") {
        room = 3;
        std::vector<std::string> es(6);
        std::vector<std::thread> th;
        for (int k = 0; k < 6; ++k) th.emplace_back([&, k] { es[k] = download(pool, (k + 1) * V + k, k, nothing); });
        for (auto& t : th) t.join();
        for (auto& x : es) e += x;
    }
    pool.leave();
    if (e.empty() && held != 0) e = "memory left after the last context";
    return e;
}
}  // namespace

int main(int argc, char** argv) {
    const std::string e = run(argc > 1 ? argv[1] : "");
    puts(e.empty() ? "ok" : e.c_str());
    return e.empty() ? 0 : 1;
}

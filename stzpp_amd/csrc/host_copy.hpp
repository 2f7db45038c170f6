// Copies between device memory and a caller's pageable host memory.
//
// The runtime's own pageable copy moves such a transfer through one thread,
// which also takes the first touch of every one of the caller's fresh pages.
// Here up to kSlots worker threads each take every kSlots-th chunk through a
// pinned slot of their own, so the transfers over the bus, the memory copies
// and the page faults of different chunks overlap.  Output cubes and the
// reference map take it; the state's fields do not.
// Measured (MI355X host, 8 threads): a 14 MB cube to the host 1.7 -> 0.67 ms
// (with one host copy less); fields of 311 MB in all to the host 31.5 -> 9.8 ms
// and of 283 MB to the device 10.2 -> 7.6 ms.  Smaller transfers stay on the runtime's path, where
// starting threads costs more than it gains: 64^3 cells (6 and 13 MB fields)
// took 2.2 ms in threads against 2.05 ms, and uploads of 9 and 18 MB 1.0 ms
// against 0.86 ms.
//
// A ring belongs to one handle: its pinned memory (16 MiB) and events are
// allocated by the first large transfer and released with the handle; the
// threads end before a call returns.
#pragma once

#include <hip/hip_runtime.h>

#include <algorithm>
#include <atomic>
#include <cstddef>
#include <cstring>
#include <exception>
#include <thread>

namespace stz {

class HostRing {
  public:
    static constexpr int kSlots = 8;
    static constexpr size_t kChunk = size_t(2) << 20;
    static constexpr size_t kDownMin = size_t(12) << 20, kUpMin = size_t(32) << 20;

    HostRing() = default;
    HostRing(const HostRing &) = delete;
    HostRing &operator=(const HostRing &) = delete;
    ~HostRing() { release(); }

    // dst (host) <- src (device), after the work enqueued on st; complete on
    // return.
    hipError_t download(void *dst, const void *src, size_t bytes, hipStream_t st) {
        if (bytes < kDownMin || !ensure()) {
            const hipError_t e = hipMemcpyAsync(dst, src, bytes, hipMemcpyDeviceToHost, st);
            return e != hipSuccess ? e : hipStreamSynchronize(st);
        }
        return run(bytes, [=](int slot, size_t at, size_t n) {
            hipError_t e = hipMemcpyAsync(pin(slot), (const char *)src + at, n, hipMemcpyDeviceToHost, st);
            if (e == hipSuccess) e = hipEventRecord(ev_[slot], st);
            if (e == hipSuccess) e = hipEventSynchronize(ev_[slot]);
            if (e == hipSuccess) std::memcpy((char *)dst + at, pin(slot), n);
            return e;
        });
    }

    // dst (device) <- src (host), enqueued on st; src may be reused on
    // return, and the copies are complete.
    hipError_t upload(void *dst, const void *src, size_t bytes, hipStream_t st) {
        if (bytes < kUpMin || !ensure()) {
            const hipError_t e = hipMemcpyAsync(dst, src, bytes, hipMemcpyHostToDevice, st);
            return e != hipSuccess ? e : hipStreamSynchronize(st);
        }
        return run(bytes, [=](int slot, size_t at, size_t n) {
            std::memcpy(pin(slot), (const char *)src + at, n);
            hipError_t e = hipMemcpyAsync((char *)dst + at, pin(slot), n, hipMemcpyHostToDevice, st);
            if (e == hipSuccess) e = hipEventRecord(ev_[slot], st);
            if (e == hipSuccess) e = hipEventSynchronize(ev_[slot]);
            return e;
        });
    }

  private:
    char *mem_ = nullptr;
    hipEvent_t ev_[kSlots] = {};
    int made_ = 0, dev_ = 0;

    char *pin(int slot) const { return mem_ + kChunk * slot; }

    // Pinned slots and events; false when they cannot be had (the caller then
    // takes the runtime's path).
    bool ensure() {
        if (mem_) return true;
        if (hipGetDevice(&dev_) == hipSuccess &&
            hipHostMalloc((void **)&mem_, kChunk * kSlots, hipHostMallocDefault) == hipSuccess) {
            while (made_ < kSlots && hipEventCreateWithFlags(&ev_[made_], hipEventDisableTiming) == hipSuccess) made_++;
            if (made_ == kSlots) return true;
        } else {
            mem_ = nullptr;
        }
        (void)hipGetLastError();
        release();
        return false;
    }

    void release() {
        for (int q = 0; q < made_; q++) (void)hipEventDestroy(ev_[q]);
        made_ = 0;
        if (mem_) (void)hipHostFree(mem_);
        mem_ = nullptr;
    }

    // move(slot, offset, size) for every chunk: chunk c in slot c mod kSlots,
    // one thread per slot (slot 0 in the calling thread).  A thread that
    // cannot be started leaves its chunks to the caller.
    template <typename F>
    hipError_t run(size_t bytes, const F &move) {
        const size_t chunks = (bytes + kChunk - 1) / kChunk;
        std::atomic<int> err{(int)hipSuccess};
        auto work = [&](int slot) {
            for (size_t c = slot; c < chunks; c += kSlots) {
                if (err.load(std::memory_order_relaxed) != (int)hipSuccess) return;
                const size_t at = c * kChunk;
                const hipError_t e = move(slot, at, std::min(kChunk, bytes - at));
                if (e != hipSuccess) err.store((int)e);
            }
        };
        std::thread th[kSlots];
        bool mine[kSlots] = {true};
        for (int s = 1; s < kSlots; s++) {
            if ((size_t)s >= chunks) break;
            try {
                th[s] = std::thread([&, s] {
                    const hipError_t e = hipSetDevice(dev_);
                    if (e != hipSuccess) err.store((int)e);
                    work(s);
                });
            } catch (const std::exception &) {  // no thread, or no memory for one
                mine[s] = true;
            }
        }
        for (int s = 0; s < kSlots; s++)
            if (mine[s]) work(s);
        for (int s = 1; s < kSlots; s++)
            if (th[s].joinable()) th[s].join();
        return (hipError_t)err.load();
    }
};

}  // namespace stz

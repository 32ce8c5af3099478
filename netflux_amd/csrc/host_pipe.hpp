// Large arrays between the caller's (pageable) memory and the device.
//
// A plain copy to or from pageable memory goes through one thread of the
// runtime: 39 GB/s up, 18 GB/s down, and 10 GB/s down into pages the caller
// has not touched yet (an array fresh from the allocator: the copying thread
// takes the page faults), where the link moves 57 GB/s.  Here a few threads,
// each with a pinned chunk of its own, copy between the caller's memory and
// their chunks while the chunks of the others are on the link.
// The state of 12.6M cells (503 MB; 8.8 ms on the link): nf_set_state 27.9 ->
// 11.3 ms (14 of them the comparison of U with U_old when both are the same
// array), nf_get_state into fresh pages 49.0 -> 12.3 ms.
//
// Not thread-safe, like the context that owns it; its pinned chunks (at most
// 32 MB) are made on the first large copy and live as long as their owner.
#pragma once
#include <hip/hip_runtime.h>

#include <algorithm>
#include <atomic>
#include <cstring>
#include <mutex>
#include <thread>
#include <vector>

namespace nf {

class HostPipe {
  public:
    HostPipe() = default;
    HostPipe(const HostPipe &) = delete;
    HostPipe &operator=(const HostPipe &) = delete;
    ~HostPipe() {
        for (Slot &q : slot_) {
            if (q.busy) (void)hipEventSynchronize(q.ev);
            (void)hipEventDestroy(q.ev);
            (void)hipHostFree(q.mem);
        }
    }

    // device -> host after the work enqueued on s so far; returns when dst holds the data
    hipError_t down(void *dst, const void *src, size_t bytes, hipStream_t s) {
        if (bytes >= MIN && ready(bytes)) return run<true>(static_cast<char *>(dst), static_cast<const char *>(src), bytes, s);
        const hipError_t e = hipMemcpyAsync(dst, src, bytes, hipMemcpyDeviceToHost, s);
        return e ? e : hipStreamSynchronize(s);
    }
    // host -> device, ordered on s; returns when src may change
    hipError_t up(void *dst, const void *src, size_t bytes, hipStream_t s) {
        if (bytes >= MIN && ready(bytes)) return run<false>(static_cast<char *>(dst), static_cast<const char *>(src), bytes, s);
        const hipError_t e = hipMemcpyAsync(dst, src, bytes, hipMemcpyHostToDevice, s);
        return e ? e : hipStreamSynchronize(s);
    }

  private:
    static constexpr size_t CHUNK = 4u << 20, MIN = 2u << 20;  // below MIN the threads cost more than they save
    static constexpr int SLOTS = 8;
    struct Slot {
        char *mem = nullptr;
        hipEvent_t ev = nullptr;
        bool busy = false;  // the event marks a copy that may still read or write mem
    };
    std::vector<Slot> slot_;

    static int slots_for(size_t bytes) {
        const int hw = (int)std::thread::hardware_concurrency();
        return (int)std::min<size_t>(std::min(SLOTS, std::max(1, hw)), (bytes + CHUNK / 2 - 1) / (CHUNK / 2));
    }
    bool ready(size_t bytes) {
        const size_t want = (size_t)slots_for(bytes);
        while (slot_.size() < want) {
            Slot q;
            if (hipHostMalloc(reinterpret_cast<void **>(&q.mem), CHUNK, hipHostMallocDefault) != hipSuccess) break;
            if (hipEventCreateWithFlags(&q.ev, hipEventDisableTiming) != hipSuccess) {
                (void)hipHostFree(q.mem);
                break;
            }
            slot_.push_back(q);
        }
        if (slot_.size() < want) (void)hipGetLastError();  // (fewer chunks, or a plain copy)
        return !slot_.empty();
    }

    template <bool DOWN>
    hipError_t run(char *dst, const char *src, size_t bytes, hipStream_t s) {
        const int T = std::min((int)slot_.size(), slots_for(bytes));
        // equal pieces of at most CHUNK, whole pages, a multiple of the threads
        const size_t rounds = (bytes + (size_t)T * CHUNK - 1) / ((size_t)T * CHUNK);
        const size_t piece = std::min(CHUNK, ((bytes + rounds * T - 1) / (rounds * T) + 4095) / 4096 * 4096);
        const size_t n = (bytes + piece - 1) / piece;
        int dev = 0;
        hipError_t e0 = hipGetDevice(&dev);
        if (e0) return e0;
        std::atomic<size_t> next{0};
        std::atomic<int> err{0};
        std::mutex mu;
        auto work = [&](int t) {
            Slot &q = slot_[t];
            hipError_t e = hipSetDevice(dev);
            while (!e && !err.load()) {
                const size_t c = next.fetch_add(1);
                if (c >= n) break;
                const size_t off = c * piece, len = std::min(piece, bytes - off);
                if (q.busy) e = hipEventSynchronize(q.ev);
                if (e) break;
                q.busy = false;
                if (!DOWN) std::memcpy(q.mem, src + off, len);
                {
                    std::lock_guard<std::mutex> lk(mu);  // the event marks this thread's copy
                    e = DOWN ? hipMemcpyAsync(q.mem, src + off, len, hipMemcpyDeviceToHost, s)
                             : hipMemcpyAsync(dst + off, q.mem, len, hipMemcpyHostToDevice, s);
                    if (!e) e = hipEventRecord(q.ev, s);
                }
                if (e) break;
                q.busy = true;
                if (DOWN) {
                    if ((e = hipEventSynchronize(q.ev))) break;
                    q.busy = false;
                    std::memcpy(dst + off, q.mem, len);
                }
            }
            if (e) err.store((int)e);
        };
        std::vector<std::thread> pool;
        try {
            pool.reserve(T);
            for (int t = 1; t < T; ++t) pool.emplace_back(work, t);
        } catch (...) {  // no more threads to be had: those there are do it
        }
        work(0);
        for (std::thread &t : pool) t.join();
        return (hipError_t)err.load();
    }
};

}  // namespace nf

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
// The pinned pieces (up to 8 of 4 MB for each device) belong to a pool: a copy
// borrows those it can get, under a lock, and returns them when its last piece
// has left; a copy that gets none is a plain one.  The pool also has a stream
// for the plain copies of many users, and the small records that kernels leave
// their results in.  It is given back with its last user.
#pragma once
#include <hip/hip_runtime.h>

#include <algorithm>
#include <atomic>
#include <cstring>
#include <map>
#include <mutex>
#include <thread>
#include <vector>

namespace nf {

class PinnedPool {
  public:
    static constexpr size_t PIECE = 4u << 20, RECORD = 128;
    struct Slot {
        char *mem = nullptr;
        hipEvent_t ev = nullptr;
        int dev = 0;
    };
    // (never destroyed: the HIP runtime may be gone when static objects are)
    static PinnedPool &get() {
        static PinnedPool *pool = new PinnedPool;
        return *pool;
    }
    void join() {
        std::lock_guard<std::mutex> lk(mu_);
        ++users_;
    }
    void leave() {
        std::lock_guard<std::mutex> lk(mu_);
        if (--users_) return;
        for (Slot &q : free_) {  // (nothing is borrowed: a user returns what it has before it leaves)
            (void)hipEventDestroy(q.ev);
            (void)hipHostFree(q.mem);
        }
        free_.clear();
        made_.clear();
        for (auto &q : copy_) (void)hipStreamDestroy(q.second);
        copy_.clear();
        for (char *p : page_) (void)hipHostFree(p);
        page_.clear();
        rec_.clear();
    }
    // a record of up to RECORD bytes, which kernels can store to on any device;
    // null if there is no memory.  (Making and freeing pinned memory of its own
    // cost a small context a quarter of its life.)
    void *record() {
        std::lock_guard<std::mutex> lk(mu_);
        try {
            if (rec_.empty()) {
                constexpr size_t PAGE = 4096;
                page_.reserve(page_.size() + 1);
                rec_.reserve((page_.size() + 1) * (PAGE / RECORD));  // giving back cannot fail
                char *p = nullptr;
                if (hipHostMalloc(reinterpret_cast<void **>(&p), PAGE, hipHostMallocPortable) != hipSuccess) {
                    (void)hipGetLastError();  // (the user does without)
                    return nullptr;
                }
                page_.push_back(p);
                for (size_t o = 0; o < PAGE; o += RECORD) rec_.push_back(p + o);
            }
        } catch (...) {
            return nullptr;
        }
        char *r = rec_.back();
        rec_.pop_back();
        return r;
    }
    void give_record(void *r) {
        std::lock_guard<std::mutex> lk(mu_);
        rec_.push_back(static_cast<char *>(r));
    }
    // A stream of device dev, which is current, for copies that are waited for;
    // null if there is none to be had, or fewer than SHARERS users: a process's
    // first four streams take 3 ms each to make, later ones 0.15, so by then this
    // one costs no more than the first copies of a user's own (HostPipe::SHARED).
    hipStream_t copy_stream(int dev) {
        std::lock_guard<std::mutex> lk(mu_);
        if (users_ < SHARERS) return nullptr;
        try {
            hipStream_t &t = copy_[dev];
            if (!t && hipStreamCreateWithFlags(&t, hipStreamNonBlocking) != hipSuccess) {
                (void)hipGetLastError();
                t = nullptr;
            }
            return t;
        } catch (...) {
            return nullptr;
        }
    }
    // up to `want` slots of device dev, which is current; make: new ones too
    std::vector<Slot> borrow(int want, int dev, bool make) {
        std::vector<Slot> got;
        std::lock_guard<std::mutex> lk(mu_);
        got.reserve(want);
        int &made = made_[dev];
        free_.reserve(SLOTS * made_.size());  // room for every slot there can be: giving back cannot fail
        for (size_t q = free_.size(); q-- > 0 && (int)got.size() < want;)
            if (free_[q].dev == dev) {
                got.push_back(free_[q]);
                free_.erase(free_.begin() + q);
            }
        while (make && (int)got.size() < want && made < SLOTS) {
            Slot s;
            s.dev = dev;
            if (hipHostMalloc(reinterpret_cast<void **>(&s.mem), PIECE, hipHostMallocDefault) != hipSuccess) break;
            if (hipEventCreateWithFlags(&s.ev, hipEventDisableTiming) != hipSuccess) {
                (void)hipHostFree(s.mem);
                break;
            }
            got.push_back(s);
            ++made;
        }
        if ((int)got.size() < want) (void)hipGetLastError();  // (fewer pieces, or a plain copy)
        return got;
    }
    void give_back(const std::vector<Slot> &s) {
        std::lock_guard<std::mutex> lk(mu_);
        free_.insert(free_.end(), s.begin(), s.end());
    }

  private:
    static constexpr int SLOTS = 8, SHARERS = 5;
    std::mutex mu_;
    std::vector<Slot> free_;
    std::vector<char *> page_, rec_;  // pages of records, free records
    std::map<int, int> made_;
    std::map<int, hipStream_t> copy_;
    int users_ = 0;
};

class HostPipe {
  public:
    HostPipe() { PinnedPool::get().join(); }
    HostPipe(const HostPipe &) = delete;
    HostPipe &operator=(const HostPipe &) = delete;
    ~HostPipe() { PinnedPool::get().leave(); }

    // device -> host after the work enqueued on s so far; returns when dst holds
    // the data.  idle: s has most likely nothing to do
    hipError_t down(void *dst, const void *src, size_t bytes, hipStream_t s, bool idle = false) {
        return copy<true>(static_cast<char *>(dst), static_cast<const char *>(src), bytes, s, idle);
    }
    // host -> device, ordered on s; src may change once s has been waited for
    hipError_t up(void *dst, const void *src, size_t bytes, hipStream_t s) {
        return copy<false>(static_cast<char *>(dst), static_cast<const char *>(src), bytes, s);
    }

  private:
    // Below this many bytes the threads cost more than they save.  Upwards the
    // runtime's own copy is at 39 GB/s and the threads' start shows for longer:
    // nf_set_state of 5.9 / 13.2 / 26.5 / 39.9 MB 215 / 413 / 775 / 1,476 us plain,
    // 271 / 506 / 795 / 1,168 through the pieces; nf_get_state of 1.9 / 3.3 / 13.2
    // MB 145 / 253 / 918 plain, 143 / 222 / 658 through them.
    static constexpr size_t CHUNK = PinnedPool::PIECE, MIN_DOWN = 2u << 20, MIN_UP = 32u << 20;
    // Pieces that are not there yet are made by a copy of at least this size, or
    // by a user's second: where memory comes in small pages making them takes
    // 1.3 ms, more than one smaller copy gains (a lone context's only nf_get_state
    // of 15.3 MB took 2.0 ms with, 1.3 without).
    static constexpr size_t MIN_MAKE = 32u << 20;
    int large_ = 0;  // copies of this user that could have made pieces

    // From this many bytes on a plain copy takes the pool's stream: a stream's
    // own first copies go through a staging buffer of 4 MB that is new to it,
    // 0.35 ms for each MB of it (set and get of 47k cells on a new context 0.79 and
    // 0.87 ms instead of 0.12 and 0.16).  It costs a second wait.
    static constexpr size_t SHARED = 256u << 10;

    static int slots_for(size_t bytes) {
        const int hw = (int)std::thread::hardware_concurrency();
        return (int)std::min<size_t>(std::min(8, std::max(1, hw)), (bytes + CHUNK / 2 - 1) / (CHUNK / 2));
    }
    template <bool DOWN>
    hipError_t copy(char *dst, const char *src, size_t bytes, hipStream_t s, bool idle = false) {
        if (bytes >= (DOWN ? MIN_DOWN : MIN_UP)) {
            int dev = 0;
            hipError_t e = hipGetDevice(&dev);
            if (e) return e;
            std::vector<PinnedPool::Slot> slot;
            const bool make = bytes >= MIN_MAKE || large_++ > 0;
            try {
                slot = PinnedPool::get().borrow(slots_for(bytes), dev, make);
            } catch (...) {  // out of memory: a plain copy
            }
            if (!slot.empty()) {
                e = run<DOWN>(slot, dev, dst, src, bytes, s);
                PinnedPool::get().give_back(slot);
                return e;
            }
        }
        const hipMemcpyKind kind = DOWN ? hipMemcpyDeviceToHost : hipMemcpyHostToDevice;
        if (bytes >= SHARED) {
            int dev = 0;
            hipError_t e = hipGetDevice(&dev);
            const hipStream_t t = e ? nullptr : PinnedPool::get().copy_stream(dev);
            if (t) {
                e = hipStreamSynchronize(s);
                if (!e) e = hipMemcpyAsync(dst, src, bytes, kind, t);
                return e ? e : hipStreamSynchronize(t);
            }
        }
        if (!DOWN) return hipMemcpyAsync(dst, src, bytes, kind, s);
        // (with nothing to wait for, the blocking copy is 3 us faster than one on s)
        if (idle) {
            const hipError_t e = hipStreamSynchronize(s);
            return e ? e : hipMemcpy(dst, src, bytes, kind);
        }
        const hipError_t e = hipMemcpyAsync(dst, src, bytes, kind, s);
        return e ? e : hipStreamSynchronize(s);
    }

    template <bool DOWN>
    hipError_t run(const std::vector<PinnedPool::Slot> &slot, int dev, char *dst, const char *src, size_t bytes,
                   hipStream_t s) {
        const int T = (int)slot.size();
        // equal pieces of at most CHUNK, whole pages, a multiple of the threads
        const size_t rounds = (bytes + (size_t)T * CHUNK - 1) / ((size_t)T * CHUNK);
        const size_t piece = std::min(CHUNK, ((bytes + rounds * T - 1) / (rounds * T) + 4095) / 4096 * 4096);
        const size_t n = (bytes + piece - 1) / piece;
        std::atomic<size_t> next{0};
        std::atomic<int> err{0};
        std::mutex mu;
        auto work = [&](int t) {
            const PinnedPool::Slot &q = slot[t];
            bool busy = false;  // the event marks a copy that may still read mem
            hipError_t e = hipSetDevice(dev);
            while (!e && !err.load()) {
                const size_t c = next.fetch_add(1);
                if (c >= n) break;
                const size_t off = c * piece, len = std::min(piece, bytes - off);
                if (busy) e = hipEventSynchronize(q.ev);
                if (e) break;
                if (!DOWN) std::memcpy(q.mem, src + off, len);
                {
                    std::lock_guard<std::mutex> lk(mu);  // the event marks this thread's copy
                    e = DOWN ? hipMemcpyAsync(q.mem, src + off, len, hipMemcpyDeviceToHost, s)
                             : hipMemcpyAsync(dst + off, q.mem, len, hipMemcpyHostToDevice, s);
                    busy = e == hipSuccess;
                    if (!e) e = hipEventRecord(q.ev, s);
                }
                if (e || !DOWN) continue;
                e = hipEventSynchronize(q.ev);
                busy = e != hipSuccess;
                if (!e) std::memcpy(dst + off, q.mem, len);
            }
            // the piece goes back to the pool: nothing may use it any more
            if (busy && hipEventSynchronize(q.ev) != hipSuccess) (void)hipStreamSynchronize(s);
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

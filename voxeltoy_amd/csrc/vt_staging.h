/*
 * vt_staging.h - large copies between pageable host memory and the device.
 *
 * The runtime's own pageable copy moves 1 MiB at a time through a staging
 * buffer, one thread copying while the device waits and the device copying
 * while the thread waits (about 90 us a MiB on an MI355X host: 20 us on the
 * link, 70 us in memcpy and page faults).  Here a ring of pinned chunks keeps
 * the link busy while several threads move the chunks to or from the caller's
 * memory.  The link is driven by a copy kernel over the pinned chunk: 2 MiB at
 * a time it moves 53 GB/s either way, the runtime's copies 24 GB/s to the
 * device and 46 GB/s from it (56 GB/s in one piece).  The kernel itself tells
 * the host that its chunk is done, by a word of pinned memory: with an event
 * after every kernel the link stood still for 5.6 us of every 45.
 *
 * A ring and its threads belong to a device, whose contexts share it: made by
 * the second large copy (the first from 16 MiB), given back when the last context is destroyed.  A copy
 * that finds both of the device's rings in use by other threads, or whose ring
 * could not be made, takes the runtime's path.
 */
#pragma once

#include <hip/hip_runtime.h>

#include <stdint.h>

#include <atomic>
#include <chrono>
#include <condition_variable>
#include <cstring>
#include <mutex>
#include <thread>
#include <vector>

namespace vt {

/* Copy kernel between device memory and a pinned chunk, both 16-byte aligned
 * (vt_volume.hip).  When all of it is copied and visible, *flag = seq; `count`
 * is a zeroed device word that the kernel leaves zero. */
hipError_t launch_copy_chunk(const void* src, void* dst, size_t bytes, uint32_t* count, uint32_t* flag, uint32_t seq,
                             hipStream_t s);

class StagingRing {
public:
    static constexpr size_t CHUNK = 2u << 20;      /* one transfer of the link */
    static constexpr size_t PIECE = 128u << 10;    /* one thread's copy */
    static constexpr int SLOTS = 6;
    static constexpr int FLAG_STRIDE = 16;         /* words: a cache line a flag */
    static constexpr int WORKERS = 3;              /* besides the calling thread */
    /* Smaller copies take the runtime's path.  Runtime / ring, us: to the device
     * 512 KiB 26 / 35, 1008 44 / 48, 2048 80 / 72; from it into fresh pages 512 34 /
     * 43, 896 53 / 55, 1008 58 / 61, 1024 (two transfers of the runtime's) 82 / 62. */
    static constexpr size_t MIN_BYTES = 1u << 20;
    static constexpr int WORKER_POLL_MS = 2, CALLER_POLL_MS = 20;
    static constexpr int PIECES = (int)(CHUNK / PIECE);

    /* Whether a copy on stream s may use the ring; it then holds `lk`.  Chunks
     * of the last write may still be on their way out of it, behind whatever
     * their stream holds: on the same stream the kernels of a read come after
     * them, a write waits for them, and other streams go without the ring. */
    bool take(std::unique_lock<std::mutex>& lk, hipStream_t s, bool to_device)
    {
        lk = std::unique_lock<std::mutex>(use_, std::try_to_lock);
        if (lk.owns_lock() && made_ && in_flight_) {
            if (stream_ == s ? to_device : hipEventQuery(last_) != hipSuccess) {
                (void)hipGetLastError();
                if (stream_ != s || hipEventSynchronize(last_) != hipSuccess) lk.unlock();
            }
            if (lk.owns_lock()) in_flight_ = false;
        }
        if (lk.owns_lock() && !make()) lk.unlock();
        return lk.owns_lock();
    }

    /* Device to host; complete when it returns. */
    hipError_t read(void* dst, const void* src, size_t bytes, hipStream_t s)
    {
        hipError_t err = hipSuccess;
        begin((char*)dst, bytes, false);
        const int n = chunks_;
        int issued = 0, arrived = 0;
        while (arrived < n && err == hipSuccess) {
            /* a slot is free again once its last chunk is out of it */
            while (issued < n && err == hipSuccess && (issued < SLOTS || copied_[issued % SLOTS].load(std::memory_order_acquire) ==
                                                                             goal(issued - SLOTS))) {
                const size_t off = (size_t)issued * CHUNK;
                if (issued >= SLOTS) copied_[issued % SLOTS].store(0, std::memory_order_relaxed);
                err = issue((const char*)src + off, slot_[issued % SLOTS], issued, s);
                if (err == hipSuccess) ++issued;
            }
            if (err != hipSuccess) break;
            if (arrived < issued && complete(arrived)) open(++arrived);
            else if (!help()) err = stalled(arrived, issued, s);
        }
        if (err != hipSuccess) abandon_.store(true, std::memory_order_release);
        finish();
        if (err != hipSuccess) (void)hipStreamSynchronize(s);
        return err;
    }

    /* Host to device, ordered on the stream; the host memory is free again
     * when it returns. */
    hipError_t write(void* dst, const void* src, size_t bytes, hipStream_t s)
    {
        hipError_t err = hipSuccess;
        begin((char*)const_cast<void*>(src), bytes, true);
        const int n = chunks_;
        int issued = 0, drained = 0;
        open(n < SLOTS ? n : SLOTS);
        while (issued < n && err == hipSuccess) {
            if (issued < open_.load(std::memory_order_relaxed) &&
                copied_[issued % SLOTS].load(std::memory_order_acquire) == goal(issued)) {
                err = issue(slot_[issued % SLOTS], (char*)dst + (size_t)issued * CHUNK, issued, s);
                if (err == hipSuccess) ++issued;
            } else if (drained < issued && open_.load(std::memory_order_relaxed) < n && complete(drained)) {
                copied_[drained % SLOTS].store(0, std::memory_order_relaxed);
                ++drained;
                open(drained + SLOTS < n ? drained + SLOTS : n);
            } else if (!help()) {
                err = stalled(drained, issued, s);
            }
        }
        if (err != hipSuccess) abandon_.store(true, std::memory_order_release);
        finish();
        if (err == hipSuccess) err = hipEventRecord(last_, s);
        if (err == hipSuccess) in_flight_ = true, stream_ = s;
        else (void)hipStreamSynchronize(s);
        return err;
    }

    /* Ends the threads and frees the ring; no copy may be running. */
    void release()
    {
        std::lock_guard<std::mutex> lk(use_);
        if (!made_) return;
        if (in_flight_) (void)hipEventSynchronize(last_);
        in_flight_ = false;
        {
            std::lock_guard<std::mutex> g(wake_lock_);
            quit_ = true;
        }
        wake_.notify_all();
        for (std::thread& t : threads_) t.join();
        threads_.clear();
        quit_ = false;
        free_slots();
        made_ = false;
    }

private:
    size_t length(int chunk) const
    {
        const size_t off = (size_t)chunk * CHUNK;
        return total_ - off < CHUNK ? total_ - off : CHUNK;
    }
    int goal(int chunk) const { return (int)((length(chunk) + PIECE - 1) / PIECE); }

    hipError_t issue(const void* from, void* to, int chunk, hipStream_t s)
    {
        seq_[chunk % SLOTS] = ++last_seq_;
        return launch_copy_chunk(from, to, length(chunk), count_, flag(chunk), last_seq_, s);
    }
    uint32_t* flag(int chunk) const { return flags_ + FLAG_STRIDE * (chunk % SLOTS); }
    bool complete(int chunk) const
    {
        return __atomic_load_n(flag(chunk), __ATOMIC_ACQUIRE) == seq_[chunk % SLOTS];
    }

    /* Nothing to copy now: chunk `waiting` is waited for.  It is polled for a
     * frame's time, since a wait that sleeps comes back later; behind longer
     * work the thread sleeps until the chunks that were issued are done. */
    hipError_t stalled(int waiting, int issued, hipStream_t s)
    {
        std::this_thread::yield();
        const auto now = std::chrono::steady_clock::now();
        if (waiting != stalled_at_) stalled_at_ = waiting, since_ = now;
        if (now - since_ < std::chrono::milliseconds(CALLER_POLL_MS) || waiting >= issued) return hipSuccess;
        const hipError_t e = hipStreamSynchronize(s);
        return e != hipSuccess ? e : complete(waiting) ? hipSuccess : hipErrorUnknown;
    }

    bool make()
    {
        if (made_) return true;
        bool ok = hipHostMalloc((void**)&flags_, SLOTS * FLAG_STRIDE * sizeof(uint32_t), hipHostMallocCoherent) == hipSuccess &&
                  hipMalloc((void**)&count_, sizeof(uint32_t)) == hipSuccess &&
                  hipEventCreateWithFlags(&last_, hipEventDisableTiming) == hipSuccess;
        for (int k = 0; k < SLOTS && ok; ++k) ok = hipHostMalloc(&slot_[k], CHUNK, hipHostMallocCoherent) == hipSuccess;
        const uint32_t zero = 0;
        ok = ok && hipMemcpy(count_, &zero, sizeof(zero), hipMemcpyHostToDevice) == hipSuccess;
        if (!ok) {
            (void)hipGetLastError();
            free_slots();
            return false;
        }
        for (int k = 0; k < SLOTS; ++k) *flag(k) = seq_[k] = 0;
        last_seq_ = 0;
        try {
            for (int k = 0; k < WORKERS; ++k) threads_.emplace_back([this] { work(); });
        } catch (...) {
            /* fewer threads copy, the caller at least */
        }
        made_ = true;
        return true;
    }

    void free_slots()
    {
        for (int k = 0; k < SLOTS; ++k) {
            if (slot_[k]) (void)hipHostFree(slot_[k]);
            slot_[k] = nullptr;
        }
        if (flags_) (void)hipHostFree(flags_);
        if (count_) (void)hipFree(count_);
        if (last_) (void)hipEventDestroy(last_);
        flags_ = count_ = nullptr;
        last_ = nullptr;
    }

    void begin(char* host, size_t bytes, bool to_ring)
    {
        host_ = host;
        total_ = bytes;
        to_ring_ = to_ring;
        chunks_ = (int)((bytes + CHUNK - 1) / CHUNK);
        pieces_ = (int64_t)((bytes + PIECE - 1) / PIECE);
        for (int k = 0; k < SLOTS; ++k) copied_[k].store(0, std::memory_order_relaxed);
        open_.store(0, std::memory_order_relaxed);
        next_.store(0, std::memory_order_relaxed);
        done_.store(0, std::memory_order_relaxed);
        abandon_.store(false, std::memory_order_relaxed);
        stalled_at_ = -1;
        {
            std::lock_guard<std::mutex> g(wake_lock_);
            ++job_;
            active_.store(true);
        }
        wake_.notify_all();
    }

    /* Wakes the workers that sleep in the job, after a sequentially consistent
     * store to open_ or active_: a worker raises asleep_ and then reads both
     * under the lock, so it is seen here or sees the store. */
    void rouse()
    {
        if (asleep_.load() == 0) return;
        { std::lock_guard<std::mutex> g(wake_lock_); }
        wake_.notify_all();
    }

    /* Chunks up to n may be copied now. */
    void open(int n)
    {
        open_.store(n);
        rouse();
    }

    /* One piece of an open chunk; false when there is none now. */
    bool help()
    {
        int64_t p = next_.load(std::memory_order_relaxed);
        for (;;) {
            if (p >= pieces_ || p / PIECES >= open_.load(std::memory_order_acquire)) return false;
            if (next_.compare_exchange_weak(p, p + 1, std::memory_order_acq_rel)) break;
        }
        const int chunk = (int)(p / PIECES);
        const size_t off = (size_t)p * PIECE;
        const size_t len = total_ - off < PIECE ? total_ - off : PIECE;
        char* ring = (char*)slot_[chunk % SLOTS] + (off - (size_t)chunk * CHUNK);
        if (to_ring_) std::memcpy(ring, host_ + off, len);
        else std::memcpy(host_ + off, ring, len);
        copied_[chunk % SLOTS].fetch_add(1, std::memory_order_acq_rel);
        done_.fetch_add(1, std::memory_order_acq_rel);
        return true;
    }

    /* every piece that was taken is copied (all of them, unless abandoned),
     * and no thread looks at the job any more: a worker raises busy_ and then
     * reads active_, both in one order with the store and the load here, so it
     * is either seen or finds the job closed.  (No lock: the workers that leave
     * would queue for it with the caller.) */
    void finish()
    {
        while (!abandon_.load(std::memory_order_acquire) && done_.load(std::memory_order_acquire) < pieces_) help();
        active_.store(false);
        rouse();
        while (busy_.load() != 0) std::this_thread::yield();
    }

    void work()
    {
        uint64_t seen = 0;
        for (;;) {
            {
                std::unique_lock<std::mutex> g(wake_lock_);
                wake_.wait(g, [&] { return quit_ || job_ != seen; });
                if (quit_) return;
                seen = job_;
                busy_.fetch_add(1);
            }
            /* Look for pieces until all are taken: with yields for a frame's
             * time, then asleep until a chunk opens (behind a render of
             * seconds every worker would keep a core busy). */
            auto last = std::chrono::steady_clock::now();
            while (active_.load() && !abandon_.load(std::memory_order_acquire) &&
                   next_.load(std::memory_order_relaxed) < pieces_) {
                if (help()) {
                    last = std::chrono::steady_clock::now();
                    continue;
                }
                std::this_thread::yield();
                if (std::chrono::steady_clock::now() - last < std::chrono::milliseconds(WORKER_POLL_MS)) continue;
                std::unique_lock<std::mutex> g(wake_lock_);
                asleep_.fetch_add(1);
                wake_.wait(g, [&] {
                    const int64_t p = next_.load(std::memory_order_relaxed);
                    return !active_.load() || p >= pieces_ || p / PIECES < open_.load();
                });
                asleep_.fetch_sub(1);
            }
            busy_.fetch_sub(1, std::memory_order_acq_rel);
        }
    }

    std::mutex use_;
    bool made_ = false, in_flight_ = false;
    void* slot_[SLOTS] = {};
    hipEvent_t last_ = nullptr;         /* after the last write, on stream_ */
    hipStream_t stream_ = nullptr;
    uint32_t* flags_ = nullptr;         /* pinned: a slot's last finished chunk */
    uint32_t* count_ = nullptr;         /* device: the copy kernel's finished workgroups */
    uint32_t seq_[SLOTS] = {}, last_seq_ = 0;
    int stalled_at_ = -1;               /* chunk that the caller waits for, since when */
    std::chrono::steady_clock::time_point since_{};
    std::vector<std::thread> threads_;
    /* the copy in progress */
    char* host_ = nullptr;
    size_t total_ = 0;
    bool to_ring_ = false;
    int chunks_ = 0;
    int64_t pieces_ = 0;
    std::atomic<int> copied_[SLOTS];
    std::atomic<int64_t> next_{ 0 }, done_{ 0 };
    std::atomic<int> open_{ 0 };
    std::atomic<bool> abandon_{ false }, active_{ false };
    std::atomic<int> busy_{ 0 };        /* workers in the job */
    std::atomic<int> asleep_{ 0 };      /* of them, waiting for a chunk */
    std::mutex wake_lock_;              /* guards the two below */
    std::condition_variable wake_;
    uint64_t job_ = 0;
    bool quit_ = false;
};

/* The copies of a device's contexts.  The second ring is for a copy that finds
 * the first in use: a read of another context may hold it behind a render. */
class Staging {
public:
    static constexpr size_t MIN_BYTES = StagingRing::MIN_BYTES;

    hipError_t read(void* dst, const void* src, size_t bytes, hipStream_t s)
    {
        std::unique_lock<std::mutex> lk;
        if (pays(bytes))
            for (StagingRing& r : ring_)
                if (r.take(lk, s, false)) return r.read(dst, src, bytes, s);
        const hipError_t e = hipMemcpyAsync(dst, src, bytes, hipMemcpyDeviceToHost, s);
        return e != hipSuccess ? e : hipStreamSynchronize(s);
    }
    hipError_t write(void* dst, const void* src, size_t bytes, hipStream_t s)
    {
        std::unique_lock<std::mutex> lk;
        if (pays(bytes))
            for (StagingRing& r : ring_)
                if (r.take(lk, s, true)) return r.write(dst, src, bytes, s);
        return hipMemcpyAsync(dst, src, bytes, hipMemcpyHostToDevice, s);
    }
    void release()
    {
        for (StagingRing& r : ring_) r.release();
        copies_.store(0, std::memory_order_relaxed);
    }

private:
    /* Making a ring and giving it back take 300 us, as much as a copy of 12 to
     * 16 MiB gains (8 MiB from the device: 0.60 ms by the runtime, 0.34 by the
     * ring, 0.76 by one made for it): a program's only copy, unless it is
     * larger, goes without. */
    static constexpr size_t ALONE_BYTES = 16u << 20;
    bool pays(size_t bytes) { return copies_.fetch_or(1, std::memory_order_relaxed) != 0 || bytes >= ALONE_BYTES; }

    StagingRing ring_[2];
    std::atomic<int> copies_{ 0 };      /* 1 after the first */
};

}  // namespace vt

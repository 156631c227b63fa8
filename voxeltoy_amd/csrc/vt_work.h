/*
 * vt_work.h - device workspace of calls that wait for their work before they
 * return.
 *
 * One buffer per device, shared by its contexts, kept from call to call (an
 * allocation and a free cost a call some 100 us and wait for the device) up to
 * KEEP bytes.  It is given back when the last context goes, and to an
 * allocation that finds no memory.  A call that finds the buffer in use, or
 * needs more, allocates for itself.
 */
#pragma once

#include <hip/hip_runtime.h>

#include <stdint.h>

#include <atomic>

namespace vt {

class DeviceWork {
public:
    static constexpr size_t KEEP = 256u << 20;

    /* Gives the buffer back unless a call uses it; whether there was one. */
    bool give_back()
    {
        if (busy_.exchange(true, std::memory_order_acquire)) return false;
        const bool had = p_ != nullptr;
        if (had) (void)hipFree(p_);
        p_ = nullptr;
        cap_ = 0;
        busy_.store(false, std::memory_order_release);
        return had;
    }

    /* hipMalloc of the caller's own memory. */
    hipError_t alloc(void** p, size_t bytes)
    {
        hipError_t e = hipMalloc(p, bytes);
        if (e != hipSuccess && give_back()) {
            (void)hipGetLastError();
            e = hipMalloc(p, bytes);
        }
        return e;
    }

private:
    friend class WorkSpace;
    /* the buffer with at least `bytes`, or null */
    uint8_t* take(size_t bytes)
    {
        if (bytes > KEEP || busy_.exchange(true, std::memory_order_acquire)) return nullptr;
        if (cap_ < bytes) {
            if (p_) (void)hipFree(p_);
            cap_ = 0;
            if (hipMalloc((void**)&p_, bytes) != hipSuccess) {
                (void)hipGetLastError();
                p_ = nullptr;
                busy_.store(false, std::memory_order_release);
                return nullptr;
            }
            cap_ = bytes;
        }
        return p_;
    }
    void leave() { busy_.store(false, std::memory_order_release); }

    std::atomic<bool> busy_{ false };
    uint8_t* p_ = nullptr;
    size_t cap_ = 0;
};

/* One call's use of it.  A call that returns early may have work on stream s
 * that still uses the memory: it is waited for unless wait() did. */
class WorkSpace {
public:
    WorkSpace(DeviceWork& w, hipStream_t s) : w_(w), s_(s) {}
    WorkSpace(const WorkSpace&) = delete;
    WorkSpace& operator=(const WorkSpace&) = delete;
    ~WorkSpace()
    {
        if (!p_) return;
        if (!waited_) (void)hipStreamSynchronize(s_);
        if (own_) (void)hipFree(p_);
        else w_.leave();
    }
    hipError_t take(size_t bytes)
    {
        p_ = w_.take(bytes);
        if (p_) return hipSuccess;
        own_ = true;
        return w_.alloc((void**)&p_, bytes);
    }
    /* The call has waited for its work. */
    void waited() { waited_ = true; }
    uint8_t* p() const { return p_; }

private:
    DeviceWork& w_;
    hipStream_t s_;
    uint8_t* p_ = nullptr;
    bool own_ = false, waited_ = false;
};

}  // namespace vt

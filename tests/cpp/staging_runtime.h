/* A device on the CPU for tests of vt_staging.h: one thread runs the copy
 * kernels of all streams in order; a stream can be kept busy for a time. */
#pragma once

#include <atomic>
#include <chrono>
#include <condition_variable>
#include <cstdlib>
#include <cstring>
#include <deque>
#include <mutex>
#include <thread>
#include <vector>

#include <hip/hip_runtime.h>

using test_clock = std::chrono::steady_clock;

struct test_stream {
    int pending = 0;                        /* guarded by test_device::lock */
    test_clock::time_point busy_until{};    /* earlier work ends then */
};
struct test_event {
    test_stream* s = nullptr;
};

struct test_device {
    struct Job {
        test_stream* s;
        const void* src;
        void* dst;
        size_t bytes;
        uint32_t* flag;
        uint32_t seq;
    };
    std::mutex lock;
    std::condition_variable more, less;
    std::deque<Job> jobs;
    bool quit = false;
    std::atomic<int> runtime_copies{ 0 }, chunks{ 0 };
    std::thread t{ [this] { run(); } };

    ~test_device()
    {
        {
            std::lock_guard<std::mutex> g(lock);
            quit = true;
        }
        more.notify_all();
        t.join();
    }
    void run()
    {
        for (;;) {
            Job j;
            {
                std::unique_lock<std::mutex> g(lock);
                for (;;) {
                    if (quit) return;
                    bool found = false;
                    for (size_t k = 0; k < jobs.size() && !found; ++k) {
                        if (test_clock::now() < jobs[k].s->busy_until) continue;
                        j = jobs[k];
                        jobs.erase(jobs.begin() + (long)k);
                        found = true;
                    }
                    if (found) break;
                    if (jobs.empty()) more.wait(g);
                    else more.wait_for(g, std::chrono::microseconds(200));
                }
            }
            std::memcpy(j.dst, j.src, j.bytes);
            __atomic_store_n(j.flag, j.seq, __ATOMIC_RELEASE);
            {
                std::lock_guard<std::mutex> g(lock);
                j.s->pending -= 1;
            }
            less.notify_all();
        }
    }
    void submit(const Job& j)
    {
        {
            std::lock_guard<std::mutex> g(lock);
            jobs.push_back(j);
            j.s->pending += 1;
        }
        chunks.fetch_add(1);
        more.notify_all();
    }
    bool idle(test_stream* s)
    {
        std::lock_guard<std::mutex> g(lock);
        return s->pending == 0 && test_clock::now() >= s->busy_until;
    }
    void wait(test_stream* s)
    {
        std::unique_lock<std::mutex> g(lock);
        while (s->pending != 0 || test_clock::now() < s->busy_until) {
            if (s->pending != 0) less.wait_for(g, std::chrono::milliseconds(2));
            else {
                const auto until = s->busy_until;
                g.unlock();
                std::this_thread::sleep_until(until);
                g.lock();
            }
        }
    }
    /* the stream has earlier work for that long */
    void keep_busy(test_stream* s, int ms)
    {
        std::lock_guard<std::mutex> g(lock);
        s->busy_until = test_clock::now() + std::chrono::milliseconds(ms);
    }
};
static test_device device_;

hipError_t hipMalloc(void** p, size_t bytes) { return *p = std::calloc(1, bytes), hipSuccess; }
hipError_t hipFree(void* p) { return std::free(p), hipSuccess; }
hipError_t hipHostMalloc(void** p, size_t bytes, unsigned) { return *p = std::calloc(1, bytes), hipSuccess; }
hipError_t hipHostFree(void* p) { return std::free(p), hipSuccess; }
hipError_t hipMemcpy(void* dst, const void* src, size_t bytes, int) { return std::memcpy(dst, src, bytes), hipSuccess; }
hipError_t hipMemcpyAsync(void* dst, const void* src, size_t bytes, int, hipStream_t s)
{
    device_.runtime_copies.fetch_add(1);
    device_.wait(s);
    std::memcpy(dst, src, bytes);
    return hipSuccess;
}
hipError_t hipStreamSynchronize(hipStream_t s) { return device_.wait(s), hipSuccess; }
hipError_t hipStreamQuery(hipStream_t s) { return device_.idle(s) ? hipSuccess : hipErrorNotReady; }
hipError_t hipEventCreateWithFlags(hipEvent_t* e, unsigned) { return *e = new test_event, hipSuccess; }
hipError_t hipEventDestroy(hipEvent_t e) { return delete e, hipSuccess; }
hipError_t hipEventRecord(hipEvent_t e, hipStream_t s) { return e->s = s, hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t e)
{
    if (e->s) device_.wait(e->s);
    return hipSuccess;
}
hipError_t hipEventQuery(hipEvent_t e) { return !e->s || device_.idle(e->s) ? hipSuccess : hipErrorNotReady; }
hipError_t hipGetLastError() { return hipSuccess; }

namespace vt {
hipError_t launch_copy_chunk(const void* src, void* dst, size_t bytes, uint32_t*, uint32_t* flag, uint32_t seq,
                             hipStream_t s)
{
    device_.submit({ s, src, dst, bytes, flag, seq });
    return hipSuccess;
}
}  // namespace vt

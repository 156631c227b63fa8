/* The ring's hand-over between the calling thread and its workers, with the
 * reordering that x86 and C++ allow: a store that is not sequentially
 * consistent may become visible only after the thread's next loads of other
 * variables.  std::atomic and std::mutex inside vt_staging.h are replaced by
 * ones that do this, pausing in between, so that what is a matter of
 * nanoseconds on a processor happens in every run.
 *
 * No worker may look at a copy that has ended, and every copy must be whole. */
#include "staging_runtime.h"

#include <cstdio>

namespace {
std::thread::id caller_;
std::atomic<bool> copying_{ false };
std::atomic<long> late_{ 0 };

struct Pending {
    void* at = nullptr;
    void (*apply)(void*, uint64_t) = nullptr;
    uint64_t value = 0;
    void drain()
    {
        if (!at) return;
        void* a = at;
        at = nullptr;
        apply(a, value);
    }
};
thread_local Pending pending_;
thread_local uint32_t dice_ = 0;

bool chance(uint32_t one_in)
{
    if (!dice_) dice_ = 2654435761u ^ (uint32_t)std::hash<std::thread::id>()(std::this_thread::get_id());
    dice_ = dice_ * 1664525u + 1013904223u;
    return (dice_ >> 8) % one_in == 0u;
}
void pause_us(int us)
{
    const auto until = test_clock::now() + std::chrono::microseconds(us);
    while (test_clock::now() < until) std::this_thread::yield();
}
}  // namespace

namespace std {
template <class T>
struct late_atomic {
    late_atomic() = default;
    late_atomic(T x) : v(x) {}
    void store(T x, memory_order o = memory_order_seq_cst)
    {
        pending_.drain();
        if (o == memory_order_seq_cst) v.store(x);
        else pending_ = { this, [](void* a, uint64_t y) { ((late_atomic*)a)->v.store((T)y); }, (uint64_t)x };
    }
    T load(memory_order = memory_order_seq_cst) const
    {
        if (sizeof(T) == 8 && this_thread::get_id() != caller_ && !copying_.load()) late_.fetch_add(1);
        if (pending_.at == this) pending_.drain();
        const T x = v.load();
        if (pending_.at) {
            if (chance(2)) pause_us(30);
            if (chance(2)) pending_.drain();            /* or it waits behind another load */
        } else if (sizeof(T) == 1 && chance(4)) {
            pause_us(50);
        }
        return x;
    }
    operator T() const { return load(); }
    T fetch_add(T x, memory_order = memory_order_seq_cst)
    {
        /* a worker that wakes at any moment of the copy */
        if (this_thread::get_id() != caller_ && chance(4)) pause_us((int)(dice_ >> 24));
        return pending_.drain(), v.fetch_add(x);
    }
    T fetch_or(T x, memory_order = memory_order_seq_cst) { return pending_.drain(), v.fetch_or(x); }
    T fetch_sub(T x, memory_order = memory_order_seq_cst) { return pending_.drain(), v.fetch_sub(x); }
    bool compare_exchange_weak(T& e, T x, memory_order = memory_order_seq_cst)
    {
        return pending_.drain(), v.compare_exchange_weak(e, x);
    }
    atomic<T> v{};
};
struct late_mutex {
    void lock() { pending_.drain(); m.lock(); }
    void unlock() { pending_.drain(); m.unlock(); }
    bool try_lock() { return pending_.drain(), m.try_lock(); }
    mutex m;
};
using late_condition_variable = condition_variable_any;
}  // namespace std

#define atomic late_atomic
#define mutex late_mutex
#define condition_variable late_condition_variable
#include "vt_staging.h"
#undef atomic
#undef mutex
#undef condition_variable

int main(int argc, char** argv)
{
    const int jobs = argc > 1 ? std::atoi(argv[1]) : 400;
    caller_ = std::this_thread::get_id();
    vt::Staging* ring = new vt::Staging();
    test_stream s;
    const size_t most = 3u << 20;
    std::vector<unsigned char> dev(most + 64), host(most + 64);
    long wrong = 0;
    for (int k = 0; k < jobs && !late_.load(); ++k) {
        const size_t bytes = (1u << 20) + (size_t)(k * 9973) % (most - (1u << 20));
        const unsigned char a = (unsigned char)(k + 1);
        std::memset(dev.data(), k & 1 ? 0xee : a, bytes);
        std::memset(host.data(), k & 1 ? a : 0xee, bytes);
        copying_.store(true);
        const hipError_t e = k & 1 ? ring->write(dev.data(), host.data(), bytes, &s) : ring->read(host.data(), dev.data(), bytes, &s);
        copying_.store(false);
        if (k % 3 == 0) pause_us(40);
        hipStreamSynchronize(&s);
        const std::vector<unsigned char>& to = k & 1 ? dev : host;
        for (size_t i = 0; i < bytes; ++i) wrong += to[i] != a;
        if (e != hipSuccess) wrong += 1;
    }
    copying_.store(true);
    ring->release();
    std::printf("late looks %ld wrong bytes %ld ring copies %d\n", late_.load(), wrong, device_.chunks.load());
    return late_.load() || wrong || device_.chunks.load() == 0;
}

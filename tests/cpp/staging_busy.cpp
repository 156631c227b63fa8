/* Copies behind a long kernel: the caller sleeps until the stream is idle, no
 * worker runs meanwhile, and the ring is free for other streams. */
#include "staging_runtime.h"
#include "vt_staging.h"

#include <cstdio>
#include <ctime>

static double cpu_s()
{
    timespec t;
    clock_gettime(CLOCK_PROCESS_CPUTIME_ID, &t);
    return (double)t.tv_sec + 1e-9 * (double)t.tv_nsec;
}

int main()
{
    constexpr int BUSY_MS = 600;
    vt::Staging* ring = new vt::Staging();
    test_stream a, b;
    const size_t bytes = 32u << 20;
    std::vector<unsigned char> da(bytes, 1), ha(bytes, 2), db(bytes, 3), hb(bytes, 4);
    ring->read(hb.data(), db.data(), bytes, &b);              /* the ring and its threads are made */
    int bad = 0;
    for (int write = 0; write < 2; ++write) {
        std::fill(ha.begin(), ha.end(), (unsigned char)(5 + write));
        std::fill(da.begin(), da.end(), (unsigned char)(7 + write));
        std::fill(hb.begin(), hb.end(), 0);
        device_.keep_busy(&a, BUSY_MS);
        const double c0 = cpu_s();
        const auto t0 = test_clock::now();
        std::thread t([&] {
            if (write) ring->write(da.data(), ha.data(), bytes, &a);
            else ring->read(ha.data(), da.data(), bytes, &a);
            hipStreamSynchronize(&a);
        });
        std::this_thread::sleep_for(std::chrono::milliseconds(BUSY_MS / 4));
        const int runtime = device_.runtime_copies.load();
        ring->read(hb.data(), db.data(), bytes, &b);
        const double other = std::chrono::duration<double>(test_clock::now() - t0).count();
        const int taken = device_.runtime_copies.load() - runtime;
        t.join();
        const double wall = std::chrono::duration<double>(test_clock::now() - t0).count(), cpu = cpu_s() - c0;
        std::printf("%s: wall %.3f cpu %.3f other stream after %.3f runtime copies %d\n", write ? "write" : "read", wall, cpu,
                    other, taken);
        bad += wall < 1e-3 * BUSY_MS || cpu > 0.5 * wall || taken != 0 || ha != da || hb != db;
    }
    ring->release();
    return bad;
}

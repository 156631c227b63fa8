/* When a device's first ring is made: not for one small copy. */
#include "staging_runtime.h"
#include "vt_staging.h"

#include <cstdio>

int main()
{
    vt::Staging* ring = new vt::Staging();
    test_stream s;
    std::vector<unsigned char> d(20u << 20, 1), h(20u << 20, 2);
    int bad = 0;
    auto copies = [&](size_t bytes, bool write) {
        const int before = device_.chunks.load();
        if (write) ring->write(d.data(), h.data(), bytes, &s);
        else ring->read(h.data(), d.data(), bytes, &s);
        hipStreamSynchronize(&s);
        bad += std::memcmp(d.data(), h.data(), bytes) != 0;
        return device_.chunks.load() - before;
    };
    for (int life = 0; life < 2; ++life) {
        bad += copies(1u << 20, false) != 0;            /* one copy of a program: the runtime's */
        bad += copies(1u << 20, true) != 1;             /* more: the ring's */
        bad += copies(5u << 20, false) != 3;
        ring->release();
    }
    bad += copies(17u << 20, true) != 9;                /* a large one at once */
    ring->release();
    bad += copies(15u << 20, false) != 0;
    ring->release();
    std::printf("bad %d\n", bad);
    return bad;
}

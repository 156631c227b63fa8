/* Sizes of a grid's tables (vt_layout.h) over extents up to 4096. */
#include "vt_layout.h"

#include <cstdio>

static long bad = 0;
static void check(bool ok, const char* what, const vt::BrickDims& d)
{
    if (ok) return;
    if (++bad < 10) std::printf("%s: %d x %d x %d\n", what, d.nx, d.ny, d.nz);
}

static void one(int nx, int ny, int nz)
{
    const vt::BrickDims d = vt::make_dims(nx, ny, nz);
    const vt::CellLayout c = vt::cell_layout(d);
    check(d.px >= d.kx + 2 && d.py >= d.ky + 2 && d.pz >= d.kz + 2, "blocks without padding", d);
    check(d.n_padded == (uint64_t)d.px * d.py * d.pz && d.n_padded < (1ull << 31), "padded blocks", d);
    const uint64_t blocks = (uint64_t)d.kx * d.ky * d.kz;
    check((uint64_t)vt::own_bit_words(d) * 32 >= blocks && (uint64_t)vt::own_bit_words(d) * 32 < blocks + 32, "own bits", d);
    const int e = 1 << c.shift;
    const uint64_t cx = (nx + e - 1) / e, cy = (ny + e - 1) / e, cz = (nz + e - 1) / e;
    check(c.ex >= cx + 2 && c.ey >= cy + 2 && c.ex % 4 == 0, "rows of cells", d);
    check(c.shift != 2 || (c.ex == (uint32_t)d.px && c.ey == (uint32_t)d.py), "cells of a block are not numbered as blocks", d);
    check((uint64_t)c.words * 16 >= (uint64_t)c.ex * c.ey * (cz + 2) && c.words % 4 == 0, "words of the codes", d);
    check((uint64_t)c.words * 4 <= vt::CODE_LDS_BYTES + 16, "codes beyond half a CU's LDS", d);
    check(c.top == 2 || c.top == 3, "top", d);
    check((1u << (c.shift + c.top)) <= 256u, "edge beyond a byte", d);
    check((c.edges() & 0xffu) == 0 && (c.edges() >> 8 & 0xffu) == (uint32_t)e - 1 &&
              (c.edges() >> 16 & 0xffu) == 2u * (uint32_t)e - 1 && (c.edges() >> 24) == ((uint32_t)e << c.top) - 1, "edges", d);
}

int main()
{
    const int some[] = { 1, 2, 3, 4, 5, 16, 63, 64, 65, 222, 224, 225, 228, 256, 263, 264, 265, 266, 512, 530, 1016, 4095, 4096 };
    for (int n = 1; n <= 4096; ++n)
        for (int a : some) {
            one(n, a, a); one(a, n, a); one(a, a, n); one(n, n, a); one(a, n, n); one(n, a, n); one(n, n, n);
        }
    std::printf("bad %ld\n", bad);
    return bad != 0;
}

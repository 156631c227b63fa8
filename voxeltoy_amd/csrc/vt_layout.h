/*
 * vt_layout.h - sizes of the tables that a grid of nx x ny x nz voxels has on
 * the device.  Plain C++, shared by the host code that allocates the tables,
 * the kernels that fill them and the CPU tests.
 */
#pragma once

#include <stdint.h>

#include <algorithm>

namespace vt {

struct BrickDims {
    int32_t nx, ny, nz;          /* voxels */
    int32_t bx, by, bz;          /* bricks per axis */
    int32_t bdim;                /* power-of-two cube edge in bricks (Morton range) */
    uint64_t n_bricks;           /* bdim^3 */
    int32_t kx, ky, kz;          /* 4x4x4 blocks per axis (ceil(n/4)) */
    /* the block grid padded by one block on every side, rows to a multiple of
     * four blocks (rows of the jump march's codes are whole bytes, and with
     * cells of one block both have one index) */
    int32_t px, py, pz;
    uint64_t n_padded;           /* px*py*pz */
};

inline BrickDims make_dims(int32_t nx, int32_t ny, int32_t nz)
{
    BrickDims d;
    d.nx = nx; d.ny = ny; d.nz = nz;
    d.bx = (nx + 7) / 8; d.by = (ny + 7) / 8; d.bz = (nz + 7) / 8;
    int32_t m = std::max(d.bx, std::max(d.by, d.bz));
    int32_t p = 1;
    while (p < m) p <<= 1;
    d.bdim = p;
    d.n_bricks = (uint64_t)p * p * p;
    d.kx = (nx + 3) / 4; d.ky = (ny + 3) / 4; d.kz = (nz + 3) / 4;
    d.px = (d.kx + 5) / 4 * 4; d.py = d.ky + 2; d.pz = d.kz + 2;
    d.n_padded = (uint64_t)d.px * d.py * d.pz;
    return d;
}

/* Grids whose renders march step by step: the jump march's error bound grows
 * with the square of the steps, and from some 700 on most jumps are undecided and
 * summed exactly.  640x400, 2 passes, 6 bounces, ms a call, jumps against steps:
 * terrain of n x n/4 x n: 800 1.91 / 2.33, 900 3.21 / 2.63, 1000 3.99 / 2.89;
 * of n x 20 x n: 800 1.60 / 1.37, 1000 2.20 / 1.54, 320x200 1500 3.00 / 1.56;
 * mesh in n^3: 600 0.77 / 1.66, 800 0.89 / 2.13. */
inline bool step_march(const BrickDims& d) { return std::max(d.nx, std::max(d.ny, d.nz)) > 900; }

/* Words of a bit per block of the grid itself. */
inline uint32_t own_bit_words(const BrickDims& d)
{
    return (uint32_t)(((uint64_t)d.kx * d.ky * d.kz + 31) / 32);
}

/* Cells of the jump march: the smallest power-of-two edge, from 4 voxels,
 * whose padded two-bit codes let two traversal workgroups share a CU's
 * 160 KiB LDS (4 up to about 266 voxels an axis, 8 up to about 530).  The
 * coded cubes are 1, 2 and 8 cells an edge, or 1, 2 and 4 where the grid has
 * at most 56 cells an axis.  Iterations a ray: 12.1 against 13.0 on a 256^3
 * terrain, 9.9 against 8.9 on a 64^3 one; the line lies below the larger of the
 * two and is not sharp, since the time hardly tells them apart.  With largest
 * cubes of 8 and of 4 cells, us a call (800x500, 4 passes, or 640x400, 2): full
 * scene 64^3 630 / 637, 128^3 746 / 739, 224^3 812 / 809, 256^3 867 / 871, 300^3
 * 1006 / 983; mesh in 512^3 579 / 578, 800^3 899 / 877; terrain of 512 977 / 975. */
struct CellLayout {
    uint32_t shift, top;         /* cells of 2^shift voxels; the largest coded cube has 2^top of them an edge */
    uint32_t ex, ey;             /* padded cells a row, rows a layer */
    uint32_t words;              /* of the codes, whole uint4 */
    /* byte c: edge of the cube of code c, minus one */
    uint32_t edges() const
    {
        return ((1u << shift) - 1u) << 8 | ((2u << shift) - 1u) << 16 | ((1u << (shift + top)) - 1u) << 24;
    }
};
constexpr uint64_t CODE_LDS_BYTES = 80640;      /* half a CU's LDS but one 1280-byte allocation unit */

inline CellLayout cell_layout(const BrickDims& d)
{
    CellLayout c;
    c.shift = 2;
    uint64_t nx, ny, nz, ex;
    for (;; ++c.shift) {
        const uint64_t e = 1ull << c.shift;
        nx = ((uint64_t)d.nx + e - 1) / e; ny = ((uint64_t)d.ny + e - 1) / e; nz = ((uint64_t)d.nz + e - 1) / e;
        /* rows of whole bytes; cells of one block are numbered as the padded
         * blocks are (the march takes a block's mask by its cell's index) */
        ex = c.shift == 2 ? (uint64_t)d.px : (nx + 5) / 4 * 4;
        c.ey = c.shift == 2 ? (uint32_t)d.py : (uint32_t)ny + 2;
        if (ex * c.ey * (nz + 2) <= CODE_LDS_BYTES * 4u) break;
    }
    c.top = std::max(nx, std::max(ny, nz)) > 56 && c.shift < 6 ? 3u : 2u;   /* an edge of at most 256: edges() holds bytes */
    c.ex = (uint32_t)ex;
    c.words = (uint32_t)((ex * c.ey * (nz + 2) + 63) / 64 * 4);
    return c;
}

}  // namespace vt

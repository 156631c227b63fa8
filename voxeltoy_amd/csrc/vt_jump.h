/*
 * vt_jump.h - the jump march of renders without statistics, and the view of
 * the grid that the marches read (gfx950).
 *
 * The march is written in terms of a few vector instructions, which the device
 * compiles to just these and the host to plain C++, so that the same source
 * marches single rays on the CPU (tests).
 */
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "vtmath.h"

namespace vt {

struct GridView {
    int32_t nx, ny, nz;
    int32_t max_steps;
    float rx, ry, rz;           /* resolution as float */
    float bmin[3], bmax[3], vs[3], ext[3];
    const uint8_t* bricks;      /* Morton bricks of 512 bytes */
    /* per-block voxel masks and non-empty bits, linear order over the block
     * grid padded by one block on every side, rows to a multiple of four
     * blocks (grid block (bx, by, bz) is padded block (bx+1, by+1, bz+1)), in
     * which every voxel outside the grid reads as occupied: the wave marches
     * stop at the first voxel outside the grid without a bounds test */
    uint32_t bxp, byp;          /* padded block extents in x and y */
    const uint64_t* occp;
    const uint32_t* bitsp;
    uint32_t bit_words_p;
    /* the bits of the grid's own blocks (x + kx (y + ky z), kx = ceil(nx / 4),
     * ...), which the megakernel stages: in LDS the padding counts.  Written
     * before each of its launches (launch_render_setup) */
    const uint32_t* bits;
    uint32_t bit_words;
    /* occp with each mask's bits reversed (voxel l of the block at bit
     * 63 - l), for the packed-coordinate march; null when an extent of the
     * grid exceeds VT_PACKED_MAX_EXTENT */
    const uint64_t* occr;
    int32_t wide;               /* padded masks span 4 GiB or more (byte offsets need 64 bits) */
    /* 2-bit empty-cube codes of the jump march, 16 per word, over the grid's
     * cells of 2^cg voxels padded by one cell on every side (rows to a multiple
     * of four cells, so that they begin at a byte; cells of one block are
     * numbered as the padded blocks), linear order (cx + ccx*(cy + ccy*cz)): 0 = some voxel of the cell is occupied or
     * outside the grid, c = 1..3 = the aligned cube of (byte c of cedge) + 1
     * voxels an edge around the cell is empty and inside the grid */
    const uint32_t* codes;
    uint32_t code_words;
    uint32_t ccx, ccy;          /* padded cell extents in x and y */
    uint32_t cg, cedge;
    float jc0;                  /* 2^-24 (2 max extent + 32): the jump march's error bound at distance 0 */
    int32_t n_emissive;
    const int32_t* emissive;    /* linear voxel indices */
    const int4* lights;         /* per emissive entry: voxel x, y, z and its material slot */
};

/* ---- vector instructions -------------------------------------------------------------- */
#if defined(__HIP_DEVICE_COMPILE__)
/* Smallest of three floats in one instruction.  The DDA's distances are
 * finite and non-negative (never NaN), where this equals fminf(fminf(a, b), c);
 * the instruction form avoids the NaN-quieting the library min inserts. */
__device__ __forceinline__ float min3f(float a, float b, float c)
{
    float r;
    asm("v_min3_f32 %0, %1, %2, %3" : "=v"(r) : "v"(a), "v"(b), "v"(c));
    return r;
}
/* middle of three; fraction; reciprocal to an ulp */
__device__ __forceinline__ float med3(float a, float b, float c) { return __builtin_amdgcn_fmed3f(a, b, c); }
__device__ __forceinline__ float fract(float v) { return __builtin_amdgcn_fractf(v); }
__device__ __forceinline__ float rcp(float v) { return __builtin_amdgcn_rcpf(v); }
/* floor, saturating; a NaN gives 0 */
__device__ __forceinline__ int32_t floor_i32(float v)
{
    int32_t r;
    asm("v_cvt_flr_i32_f32 %0, %1" : "=v"(r) : "v"(v));
    return r;
}
/* -1 when bit (at & 31) of v is set, else 0 */
__device__ __forceinline__ int32_t bit_mask(uint32_t v, uint32_t at)
{
    int32_t r;
    asm("v_bfe_i32 %0, %1, %2, 1" : "=v"(r) : "v"(v), "v"(at));
    return r;
}
/* (x & 3) + 4 (y & 3) + 16 (z & 3): a voxel's bit in its block's mask */
__device__ __forceinline__ uint32_t local_bit(uint32_t vx, uint32_t vy, uint32_t vz)
{
    uint32_t b = vy << 2;
    asm("v_bfi_b32 %0, 3, %1, %2" : "=v"(b) : "v"(vx), "v"(b));
    uint32_t c = vz << 4;
    asm("v_bfi_b32 %0, 15, %1, %2" : "=v"(c) : "v"(b), "v"(c));
    return c & 63u;
}
/* (a ^ b) + c; c is wave-uniform with UNI */
template <bool UNI>
__device__ __forceinline__ uint32_t xor_add(int32_t a, int32_t b, uint32_t c)
{
    uint32_t r;
    if constexpr (UNI) asm("v_xad_u32 %0, %1, %2, %3" : "=v"(r) : "v"(a), "v"(b), "s"(c));
    else asm("v_xad_u32 %0, %1, %2, %3" : "=v"(r) : "v"(a), "v"(b), "v"(c));
    return r;
}
/* W bits of v from bit (at & 31); v is wave-uniform with UNI */
template <uint32_t W, bool UNI>
__device__ __forceinline__ uint32_t field(uint32_t v, uint32_t at)
{
    uint32_t r;
    if constexpr (UNI) asm("v_bfe_u32 %0, %1, %2, %3" : "=v"(r) : "s"(v), "v"(at), "n"(W));
    else asm("v_bfe_u32 %0, %1, %2, %3" : "=v"(r) : "v"(v), "v"(at), "n"(W));
    return r;
}
/* x + ex (y + ey z) on 24-bit operands; ex and ey are wave-uniform with UNI */
template <bool UNI>
__device__ __forceinline__ uint32_t index3(uint32_t ix, uint32_t iy, uint32_t iz, uint32_t ex, uint32_t ey)
{
    uint32_t r;
    if constexpr (UNI) {
        asm("v_mad_u32_u24 %0, %1, %2, %3" : "=v"(r) : "v"(iz), "s"(ey), "v"(iy));
        asm("v_mad_u32_u24 %0, %1, %2, %3" : "=v"(r) : "v"(r), "s"(ex), "v"(ix));
    } else {
        asm("v_mad_u32_u24 %0, %1, %2, %3" : "=v"(r) : "v"(iz), "v"(ey), "v"(iy));
        asm("v_mad_u32_u24 %0, %1, %2, %3" : "=v"(r) : "v"(r), "v"(ex), "v"(ix));
    }
    return r;
}
/* a word of the codes; UNI: from the start of the workgroup's LDS, where they
 * are (an address of its own would cost an add) */
template <bool UNI>
__device__ __forceinline__ uint32_t code_word(const uint32_t* codes, uint32_t i)
{
    if constexpr (UNI) return *(const __attribute__((address_space(3))) uint32_t*)(i << 2);
    else return ((const __attribute__((address_space(1))) uint32_t*)codes)[i];
}
/* a block's voxel mask */
__device__ __forceinline__ uint64_t load_mask(const uint64_t* occp, uint32_t i)
{
    return ((const __attribute__((address_space(1))) uint64_t*)occp)[i];
}
__device__ __forceinline__ int lanes_with(bool p) { return __popcll(__builtin_amdgcn_ballot_w64(p)); }
#else
/* The host's equivalents, for one ray. */
__device__ __forceinline__ float min3f(float a, float b, float c) { return fminf(fminf(a, b), c); }
__device__ __forceinline__ float med3(float a, float b, float c) { return fmaxf(fminf(a, b), fminf(fmaxf(a, b), c)); }
__device__ __forceinline__ float fract(float v) { return fminf(v - floorf(v), 0x1.fffffep-1f); }
__device__ __forceinline__ float rcp(float v) { return 1.0f / v; }
__device__ __forceinline__ int32_t floor_i32(float v)
{
    const float f = floorf(v);
    return f != f ? 0 : f >= 2147483648.0f ? INT32_MAX : f < -2147483648.0f ? INT32_MIN : (int32_t)f;
}
__device__ __forceinline__ int32_t bit_mask(uint32_t v, uint32_t at) { return -(int32_t)((v >> (at & 31u)) & 1u); }
__device__ __forceinline__ uint32_t local_bit(uint32_t vx, uint32_t vy, uint32_t vz)
{
    return (vx & 3u) | ((vy & 3u) << 2) | ((vz & 3u) << 4);
}
template <bool UNI>
__device__ __forceinline__ uint32_t xor_add(int32_t a, int32_t b, uint32_t c) { return (uint32_t)(a ^ b) + c; }
template <uint32_t W, bool UNI>
__device__ __forceinline__ uint32_t field(uint32_t v, uint32_t at) { return (v >> (at & 31u)) & ((1u << W) - 1u); }
template <bool UNI>
__device__ __forceinline__ uint32_t index3(uint32_t ix, uint32_t iy, uint32_t iz, uint32_t ex, uint32_t ey)
{
    return ix + (ex & 0xffffffu) * ((iy + (ey & 0xffffffu) * (iz & 0xffffffu)) & 0xffffffu);
}
template <bool UNI>
__device__ __forceinline__ uint32_t code_word(const uint32_t* codes, uint32_t i) { return codes[i]; }
__device__ __forceinline__ uint64_t load_mask(const uint64_t* occp, uint32_t i) { return occp[i]; }
__device__ __forceinline__ int lanes_with(bool p) { return p ? 1 : 0; }
#endif

/* ---- jump march ------------------------------------------------------------------------
 * The voxel at which the DDA of dda.h:7-61 stops, without its step count:
 * the traversal of renders that collect no statistics.
 *
 * The DDA visits voxels in the order of three sequences, one per axis: X_0 =
 * dis.x and X_{k+1} = fl(X_k + a.x) (a = |1/d|), the value at which the k-th
 * x step is taken, and the same for y and z.  Each iteration takes the axes
 * whose next value is the smallest, so the position after all values <= m
 * depends on m alone: x0 + #{k: X_k <= m}, and so on.  While the ray is inside an
 * aligned cube of empty voxels the visited voxels need no test, and the whole
 * passage is one jump: m = the smallest of the three values at which an axis
 * steps out of the cube, then the three counts.
 *
 * Values and counts are evaluated on the real line X_0 + k a.  Every add of
 * the FP32 sums is off by at most half an ulp, so with M = m / (smallest a) the
 * two sequences that a decision compares are together off their lines by at
 * most 2^-24 (M^2 + 3M) steps, and the evaluation itself by 2^-24 (3M + 2
 * extent + 8); del = 2^-24 (1.06 (M + 4)^2 + 2 extent + 32) covers both.
 * With q the real-valued position (an integer where an axis steps), floor(q +
 * del) is the exact position unless q lies within del of an integer; on the
 * axis that leaves the cube it always does, and it is then right as well as
 * long as del stays below 1 (3970 steps).  When a second axis is that near an integer the order of the
 * two steps is undecided (0.1-0.3 % of the jumps).  Both orders and a common
 * step end in the same voxel, by way of one of the two voxels where one of the
 * steps is still missing: if both are empty the ray passes and the order does
 * not matter.  That holds when no other step can fall between the two, which
 * are at most 2 del a apart (a: the longer step of the two axes): the third
 * axis must be 2 del (1 + a / its step) from an integer on either side.
 * jump() leaves such a jump to near_jump(), which leaves the rest (10-19 % of
 * the undecided jumps) to resolve(), which compares the FP32 sums themselves.
 *
 * Axes are mirrored (x ^ -1) so that every step is +1 and the far face of an
 * aligned cube is x | (edge - 1).  A ray whose set-up leaves the range of the
 * limits below (non-finite or far from unit directions) is marched step by
 * step instead.
 *
 * In a cell with an occupied voxel the cube is the aligned 2x2x2 around the
 * position when the mask shows it empty: 42 % of the iterations are in such
 * cells, and one shift and one AND there save 12-15 % of all iterations.
 *
 * Full-shading scene (256^3, 99 DDA steps a ray): 10.7 iterations a ray (12.1
 * without the cubes of 2), 99.9 % of the rays within 56 (69; the steps: 580). */
#define VT_JUMP_A_MIN 9.765625e-4f        /* 2^-10 */
#define VT_JUMP_A_MAX 2.0e5f
#define VT_ULP24 5.9604644775390625e-8f   /* 2^-24 */
/* GridView::jc0 of a grid whose longest axis has n voxels */
__host__ __device__ __forceinline__ float jump_bound0(int32_t n) { return VT_ULP24 * (float)(2 * n + 32); }
/* 1.03 * 2^-12 and 4 times that: (m / a W1 + W4)^2 = 1.06 * 2^-24 (m / a + 4)^2 */
#define VT_JUMP_W1 2.5146484375e-4f
#define VT_JUMP_W4 1.005859375e-3f

/* The sum X + a + a + ... of n FP32 adds, exactly.  Inside one binade every
 * add rounds a to the same multiple of the ulp (once the sum is the result of
 * an add there, which settles the parity of ties), so a run of adds that stays
 * below the binade's end is one exact multiply-add. */
__device__ __forceinline__ float sum_steps(float X, float a, float ia, int32_t n)
{
    while (n > 0) {
        const float p = X + a;
        if (--n == 0) return p;
        X = p + a;
        --n;
        const uint32_t ub = __float_as_uint(X) & 0x7f800000u;
        if (n > 0 && ub == (__float_as_uint(p) & 0x7f800000u)) {
            const float end = __uint_as_float(ub + 0x00800000u);
            /* two steps short of the end: covers the rounding of the quotient
             * and, over at most 4096 adds, of a */
            int32_t r = (int32_t)((end - X) * ia) - 2;
            r = r < n ? r : n;
            if (r > 0) {
                X = __builtin_fmaf((float)r, (X + a) - X, X);
                n -= r;
            }
        }
    }
    return X;
}

struct JumpState {
    int32_t x, y, z;            /* mirrored position */
    int32_t x0, y0, z0;         /* mirrored start */
    int32_t fx, fy, fz;         /* 0, or -1 on a mirrored axis */
    float X0, Y0, Z0, ax, ay, az, ix, iy, iz, q_x, q_y, q_z;
    float w1;                   /* W1 over the smallest a */

    /* the error bound at value m, in steps */
    __device__ __forceinline__ float bound(const GridView& g, float m) const
    {
        const float w = __builtin_fmaf(m, w1, VT_JUMP_W4);
        return __builtin_fmaf(w, w, g.jc0);
    }

    enum { OUTSIDE = 0, READY = 1, STEPWISE = 2 };

    /* DdaState::init's arithmetic from a queue entry (queue_a, queue_b): the
     * distance to the first step is |1/d| times the part of the voxel that is
     * left along the ray, in [0, 1].  STEPWISE when the bound does not hold;
     * compared as integers, a NaN exceeds every limit. */
    __device__ __forceinline__ int init(const GridView& g, float4 qa, float2 qb)
    {
        const float vox = ((qa.x - g.bmin[0]) * g.ext[0]) * g.rx;
        const float voy = ((qa.y - g.bmin[1]) * g.ext[1]) * g.ry;
        const float voz = ((qa.z - g.bmin[2]) * g.ext[2]) * g.rz;
        const float bx = floorf(vox), by = floorf(voy), bz = floorf(voz);
        /* saturating, a NaN gives 0 and is found below */
        const int32_t jx = floor_i32(vox), jy = floor_i32(voy), jz = floor_i32(voz);
        if ((uint32_t)jx >= (uint32_t)g.nx || (uint32_t)jy >= (uint32_t)g.ny || (uint32_t)jz >= (uint32_t)g.nz)
            return OUTSIDE;
        ax = vt_absf(qa.w); ay = vt_absf(qb.x); az = vt_absf(qb.y);
        X0 = vt_absf(((bx - vox) + 0.5f) + __builtin_copysignf(0.5f, qa.w)) * ax;
        Y0 = vt_absf(((by - voy) + 0.5f) + __builtin_copysignf(0.5f, qb.x)) * ay;
        Z0 = vt_absf(((bz - voz) + 0.5f) + __builtin_copysignf(0.5f, qb.y)) * az;
        const uint32_t ua = __float_as_uint(ax), ub = __float_as_uint(ay), uc = __float_as_uint(az);
        const uint32_t u0 = __float_as_uint(X0), u1 = __float_as_uint(Y0), u2 = __float_as_uint(Z0);
        const uint32_t lo = min(min(ua, ub), uc), hi = max(max(ua, ub), uc), h0 = max(max(u0, u1), u2);
        if (lo < __float_as_uint(VT_JUMP_A_MIN) || max(hi, h0) > __float_as_uint(VT_JUMP_A_MAX)) return STEPWISE;
        fx = (int32_t)__float_as_uint(qa.w) >> 31;
        fy = (int32_t)__float_as_uint(qb.x) >> 31;
        fz = (int32_t)__float_as_uint(qb.y) >> 31;
        x = x0 = jx ^ fx; y = y0 = jy ^ fy; z = z0 = jz ^ fz;
        ix = rcp(ax); iy = rcp(ay); iz = rcp(az);
        w1 = VT_JUMP_W1 * fmaxf(fmaxf(ix, iy), iz);
        q_x = __builtin_fmaf(-X0, ix, (float)(x0 + 1));
        q_y = __builtin_fmaf(-Y0, iy, (float)(y0 + 1));
        q_z = __builtin_fmaf(-Z0, iz, (float)(z0 + 1));
        return READY;
    }

    /* Edge minus one of the empty aligned cube around the position, 0 for a
     * single voxel; -1 when the voxel is occupied or outside the grid.
     * FINE: cells are the 4x4x4 blocks.  UNI: one grid for the whole wave. */
    template <bool FINE, bool UNI>
    __device__ __forceinline__ int32_t lookup(const GridView& g) const
    {
        const uint32_t cg = FINE ? 2u : g.cg;
        const uint32_t pad = 1u << cg;
        const uint32_t ux = xor_add<UNI>(x, fx, pad), uy = xor_add<UNI>(y, fy, pad), uz = xor_add<UNI>(z, fz, pad);
        const uint32_t ci = index3<UNI>(ux >> cg, uy >> cg, uz >> cg, g.ccx, g.ccy);
        const uint32_t word = code_word<UNI>(g.codes, ci >> 4);
        const uint32_t c = field<2, false>(word, ci << 1);
        int32_t edge = (int32_t)field<8, UNI>(g.cedge, c << 3);
        if (c == 0u) {
            uint32_t bi = ci;
            if (!FINE) {
                const uint32_t k = pad - 4u;
                bi = index3<UNI>((ux - k) >> 2, (uy - k) >> 2, (uz - k) >> 2, g.bxp, g.byp);
            }
            const uint64_t m = load_mask(g.occp, bi);
            /* the 2x2x2 voxels around the position, then the voxel itself */
            const uint32_t b = local_bit(ux, uy, uz);
            const uint32_t t = (uint32_t)(m >> (b & 0x2au));
            edge = (t & 0x00330033u) == 0u ? 1 : 0;
            if (!FINE && m == 0ull) edge = 3;
            edge |= bit_mask(t, b & 0x15u);
        }
        return edge;
    }

    /* Whether the voxel at mirrored (px, py, pz), inside the grid or one past
     * it, is occupied or outside the grid. */
    template <bool UNI>
    __device__ __forceinline__ bool blocked(const GridView& g, int32_t px, int32_t py, int32_t pz) const
    {
        const uint32_t vx = xor_add<false>(px, fx, 4u), vy = xor_add<false>(py, fy, 4u), vz = xor_add<false>(pz, fz, 4u);
        const uint64_t m = load_mask(g.occp, index3<UNI>(vx >> 2, vy >> 2, vz >> 2, g.bxp, g.byp));
        return ((m >> local_bit(vx, vy, vz)) & 1ull) != 0ull;
    }

    /* Leave the cube of lookup(); false, with the position unchanged, when
     * there is none or a second axis is within the bound of a step. */
    __device__ __forceinline__ bool jump(const GridView& g, int32_t edge)
    {
        float px, py, pz;
        const float del2 = 2.0f * leave(g, edge, px, py, pz);
        const float r = med3(fract(px), fract(py), fract(pz));
        const bool ok = (int)!(r < del2) & (int)(edge >= 0);
        if (ok) {
            x = floor_i32(px); y = floor_i32(py); z = floor_i32(pz);
        }
        return ok;
    }

    /* The position (plus the bound, which it returns) at the value that leaves
     * the cube. */
    __device__ __forceinline__ float leave(const GridView& g, int32_t edge, float& px, float& py, float& pz) const
    {
        const int32_t bx = x | edge, by = y | edge, bz = z | edge;
        const float m = min3f(__builtin_fmaf((float)(bx - x0), ax, X0), __builtin_fmaf((float)(by - y0), ay, Y0),
                              __builtin_fmaf((float)(bz - z0), az, Z0));
        const float del = bound(g, m);
        px = __builtin_fmaf(m, ix, q_x) + del;
        py = __builtin_fmaf(m, iy, q_y) + del;
        pz = __builtin_fmaf(m, iz, q_z) + del;
        return del;
    }

    /* The jump that jump() declined: false, with the position unchanged, when
     * the order of two steps is undecided and matters. */
    template <bool UNI>
    __device__ __forceinline__ bool near_jump(const GridView& g, int32_t edge)
    {
        float px, py, pz;
        const float del2 = 2.0f * leave(g, edge, px, py, pz);
        const float rx = fract(px), ry = fract(py), rz = fract(pz);
        const int32_t tx = floor_i32(px), ty = floor_i32(py), tz = floor_i32(pz);
        /* steps ahead only: one that is behind was taken before */
        const bool mx = tx > x, my = ty > y, mz = tz > z;
        const bool nx = rx < del2 && mx, ny = ry < del2 && my, nz = rz < del2 && mz;
        /* a bound near 1 (from about 3860 steps) no longer tells the step that
         * leaves the cube from the one after it */
        if ((nx && ny && nz) || del2 > 1.9f) return false;
        if ((nx && ny) || (ny && nz) || (nz && nx)) {
            const float am = fmaxf(fmaxf(nx ? ax : 0.0f, ny ? ay : 0.0f), nz ? az : 0.0f);
            const float ex = del2 * __builtin_fmaf(am, ix, 1.0f), ey = del2 * __builtin_fmaf(am, iy, 1.0f),
                        ez = del2 * __builtin_fmaf(am, iz, 1.0f);
            if (!(fmaxf(fmaxf(ex, ey), ez) < 0.4f)) return false;
            if ((!nx && ((mx && rx < ex) || rx > 1.0f - ex)) || (!ny && ((my && ry < ey) || ry > 1.0f - ey)) ||
                (!nz && ((mz && rz < ez) || rz > 1.0f - ez)))
                return false;
            /* the voxels where one of the two steps is missing */
            if (nx && blocked<UNI>(g, tx - 1, ty, tz)) return false;
            if (ny && blocked<UNI>(g, tx, ty - 1, tz)) return false;
            if (nz && blocked<UNI>(g, tx, ty, tz - 1)) return false;
        }
        x = tx; y = ty; z = tz;
        return true;
    }

    /* The jump that near_jump() left undecided: the smallest value that leaves the
     * cube from the FP32 sums, then on each axis the steps up to it, the last
     * one checked against its sum where the real line leaves it open. */
    __device__ __forceinline__ void resolve(const GridView& g, int32_t edge)
    {
        const int32_t at[3] = { x, y, z }, s0[3] = { x0, y0, z0 };
        const float S0[3] = { X0, Y0, Z0 }, a[3] = { ax, ay, az }, ia[3] = { ix, iy, iz }, q[3] = { q_x, q_y, q_z };
        float t[3], m = __uint_as_float(0x7f800000u);
#pragma unroll
        for (int k = 0; k < 3; ++k) {
            t[k] = __builtin_fmaf((float)((at[k] | edge) - s0[k]), a[k], S0[k]);
            m = fminf(m, t[k]);
        }
        /* an axis further behind than both errors leaves later */
        const float m0 = m, d0 = 2.0f * bound(g, m);
        const float first = m0 == t[0] ? a[0] : m0 == t[1] ? a[1] : a[2];
        m = __uint_as_float(0x7f800000u);
#pragma unroll
        for (int k = 0; k < 3; ++k)
            if (t[k] - m0 <= d0 * (a[k] + first)) m = fminf(m, sum_steps(S0[k], a[k], ia[k], (at[k] | edge) - s0[k]));
        const float del = bound(g, m);
        int32_t to[3];
#pragma unroll
        for (int k = 0; k < 3; ++k) {
            const float p = __builtin_fmaf(m, ia[k], q[k]) + del;
            to[k] = floor_i32(p);
            /* at most one step too far unless the bound is above 1/2 (more
             * than 2800 steps) */
            if (fract(p) < del + del)
                while (to[k] > at[k] && sum_steps(S0[k], a[k], ia[k], to[k] - 1 - s0[k]) > m) to[k] -= 1;
        }
        x = to[0]; y = to[1]; z = to[2];
    }

    __device__ __forceinline__ int32_t gx() const { return x ^ fx; }
    __device__ __forceinline__ int32_t gy() const { return y ^ fy; }
    __device__ __forceinline__ int32_t gz() const { return z ^ fz; }
};

/* The jump march of the wave's `live` lanes: at most `jumps` jumps, until
 * fewer than `keep` of them still march.  A lane is live no longer at its
 * ray's last voxel (edge -1), or where leaving the cube of `edge` needs more
 * than JumpState::jump.  The loop is the whole wave's, with one mask: lanes that
 * leave it one by one make the compiler copy the position twice in every
 * iteration, and every further flag costs a merge. */
template <bool FINE, bool UNI>
__device__ __forceinline__ void jump_march(JumpState& J, const GridView& g, int jumps, int keep, bool& live, int32_t& edge)
{
    do {
        if (live) {
            edge = J.lookup<FINE, UNI>(g);
            live = J.jump(g, edge);
        }
    } while (--jumps > 0 && lanes_with(live) >= keep);
}

}  // namespace vt

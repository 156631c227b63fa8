/*
 * vt_volume.hip - grid layout conversion and the triangle voxelizer.
 *
 * The voxelizer kernel restates voxelize.vs (:20-28) and voxelize.gs
 * (swizzleTri :83-137, voxelizeTriPostSwizzle :146-260, main :262-279) with
 * one thread per triangle; covered voxels are written straight into the
 * Morton-bricked grid (and optionally into a dense byte image).  Duplicate
 * writes of the same value by neighbouring triangles are the same benign
 * race the geometry shader has (voxelize.gs:142).
 */
#include "vt_kernels.h"
#include "vt_staging.h"

namespace vt {

__device__ __forceinline__ uint64_t brick_byte(int32_t x, int32_t y, int32_t z)
{
    return (uint64_t)brick_morton((uint32_t)x >> 3, (uint32_t)y >> 3, (uint32_t)z >> 3) * 512u +
           local_morton((uint32_t)x, (uint32_t)y, (uint32_t)z);
}

/* One coalesced pass over the offsets (64 MB in 17 us).  With the conversion
 * below it replaces three loops over the grid on one host thread: loading a
 * 256^3 grid of offsets and rendering 960x540 from it went from 7.7 to 2.2 ms,
 * 1.3 of them the link. */
__global__ __launch_bounds__(256) void scan_offsets_kernel(const int32_t* __restrict__ dense, uint64_t n, int32_t lut_n,
                                                           uint8_t* used, unsigned long long* bad)
{
    const uint64_t n4 = n / 4u;
    int32_t last = -1;                       /* neighbours mostly share an offset or are empty */
    uint64_t first_bad = ~0ull;
    auto look = [&](int32_t o, uint64_t i) {
        if (o < 0 || o == last) return;
        last = o;
        if (o >= lut_n) first_bad = i < first_bad ? i : first_bad, last = -1;
        else if (!used[o]) used[o] = 1u;
    };
    for (uint64_t q = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; q < n4; q += (uint64_t)gridDim.x * blockDim.x) {
        const int4 v = ((const int4*)dense)[q];
        look(v.x, 4u * q);
        look(v.y, 4u * q + 1u);
        look(v.z, 4u * q + 2u);
        look(v.w, 4u * q + 3u);
    }
    if (blockIdx.x == 0 && threadIdx.x < (n & 3u)) look(dense[4u * n4 + threadIdx.x], 4u * n4 + threadIdx.x);
    if (first_bad != ~0ull) atomicMin(bad, (unsigned long long)first_bad);
}

__global__ __launch_bounds__(256) void check_emissive_kernel(const int32_t* __restrict__ emissive, int32_t n,
                                                             uint64_t n_vox, const int32_t* __restrict__ offsets,
                                                             const uint8_t* __restrict__ ids,
                                                             const uint8_t* __restrict__ remap, uint32_t* bad)
{
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x) {
        const int32_t e = emissive[i];
        const bool ok = e >= 0 && (uint64_t)e < n_vox && (offsets ? offsets[e] >= 0 : remap[ids[e]] != 0u);
        if (!ok) atomicMin(bad, (uint32_t)i);
    }
}

/* Four flags (bits 0..3) of the non-zero bytes of v. */
__device__ __forceinline__ uint32_t nonzero_bytes(uint32_t v)
{
    const uint32_t t = (((v & 0x7f7f7f7fu) + 0x7f7f7f7fu) | v) & 0x80808080u;
    return ((t >> 7) * 0x10204080u) >> 28;
}

/* One thread per 4x4x4 block of the padded block grid, consecutive threads
 * along x.  A block's 64 slots are one Morton-ordered 64-byte line of its
 * brick: dword z0 + 2 x1 + 4 y1 + 8 z1 holds the voxels (x0, y0) of a 2x2
 * square.  From a dense grid (SRC 1 offsets, 2 ids) a thread reads the block's
 * 16 rows of four voxels (a wave's rows are contiguous), writes the line and
 * forms the mask from the same registers, so the grid is read once and the
 * bricks are not read back.  Voxels outside the grid are set in the masks, the
 * padding's masks are all set.  Bound by memory: 256^3 offsets (64 MB read, 21
 * MB written) in 27 us, where the conversion into bricks alone took 68 and the
 * padded masks and two passes of bits 25 more.  From the bricks 5 us (512^3,
 * 35; the masks alone took 48 and 30 for two separate layouts). */
template <int SRC>
__global__ __launch_bounds__(256) void blocks_kernel(BrickDims d, const void* __restrict__ dense,
                                                     const uint8_t* __restrict__ lut, uint8_t* __restrict__ bricks,
                                                     BlockLevels L)
{
    const uint32_t px = (uint32_t)d.px, py = (uint32_t)d.py;
    const uint32_t n = (uint32_t)d.n_padded;  /* at most 1028 * 1026^2 */
    const bool rows4 = (d.nx & 3) == 0;       /* every row of four voxels aligned */
    for (uint32_t base = blockIdx.x * blockDim.x; base < n; base += gridDim.x * blockDim.x) {
        const uint32_t w = base + threadIdx.x;
        const uint32_t r = w / px, bx = w - r * px;
        const uint32_t bz = r / py, by = r - bz * py;
        uint64_t m = ~0ull;
        if (w < n && bx - 1u < (uint32_t)d.kx && by - 1u < (uint32_t)d.ky && bz - 1u < (uint32_t)d.kz) {
            const uint32_t gx = bx - 1u, gy = by - 1u, gz = bz - 1u;
            const int32_t x0 = (int32_t)(4u * gx), y0 = (int32_t)(4u * gy), z0 = (int32_t)(4u * gz);
            uint4* line = (uint4*)(bricks + (uint64_t)brick_morton(gx >> 1, gy >> 1, gz >> 1) * 512u +
                                   ((gx & 1u) | ((gy & 1u) << 1) | ((gz & 1u) << 2)) * 64u);
            m = 0ull;
            if (SRC == 0) {
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    const uint4 v = line[q];
                    const uint32_t wd[4] = { v.x, v.y, v.z, v.w };
#pragma unroll
                    for (int k = 0; k < 4; ++k) {
                        const int i = 4 * q + k;
                        const uint32_t f = nonzero_bytes(wd[k]);
                        m |= (uint64_t)((f & 3u) | ((f & 12u) << 2))
                             << (2 * ((i >> 1) & 1) + 8 * ((i >> 2) & 1) + 16 * ((i & 1) + 2 * (i >> 3)));
                    }
                }
            } else {
                uint32_t row[16];             /* slots of row (y, z) at 4 z + y */
#pragma unroll
                for (int i = 0; i < 16; ++i) {
                    const int32_t y = y0 + (i & 3), z = z0 + (i >> 2);
                    row[i] = 0u;
                    if (y >= d.ny || z >= d.nz) continue;
                    const uint64_t at = (uint64_t)x0 + (uint64_t)d.nx * ((uint64_t)y + (uint64_t)d.ny * (uint64_t)z);
                    if (SRC == 1) {
                        const int32_t* p = (const int32_t*)dense + at;
                        int32_t o[4] = { -1, -1, -1, -1 };
                        if (rows4) {
                            const int4 v = *(const int4*)p;
                            o[0] = v.x; o[1] = v.y; o[2] = v.z; o[3] = v.w;
                        } else {
#pragma unroll
                            for (int k = 0; k < 4; ++k)
                                if (x0 + k < d.nx) o[k] = p[k];
                        }
#pragma unroll
                        for (int k = 0; k < 4; ++k)
                            if (o[k] >= 0) row[i] |= (uint32_t)lut[o[k]] << (8 * k);
                    } else {
                        const uint8_t* p = (const uint8_t*)dense + at;
                        if (rows4) {
                            const uint32_t v = *(const uint32_t*)p;
#pragma unroll
                            for (int k = 0; k < 4; ++k) row[i] |= (uint32_t)lut[(v >> (8 * k)) & 0xffu] << (8 * k);
                        } else {
#pragma unroll
                            for (int k = 0; k < 4; ++k)
                                if (x0 + k < d.nx) row[i] |= (uint32_t)lut[p[k]] << (8 * k);
                        }
                    }
                    m |= (uint64_t)nonzero_bytes(row[i]) << (4 * (i & 3) + 16 * (i >> 2));
                }
                uint32_t out[16];
#pragma unroll
                for (int i = 0; i < 16; ++i) {
                    const int x1 = (i >> 1) & 1, y1 = (i >> 2) & 1, z = (i & 1) + 2 * (i >> 3);
                    out[i] = ((row[4 * z + 2 * y1] >> (16 * x1)) & 0xffffu) |
                             (((row[4 * z + 2 * y1 + 1] >> (16 * x1)) & 0xffffu) << 16);
                }
#pragma unroll
                for (int q = 0; q < 4; ++q) line[q] = make_uint4(out[4 * q], out[4 * q + 1], out[4 * q + 2], out[4 * q + 3]);
            }
            if (x0 + 4 > d.nx || y0 + 4 > d.ny || z0 + 4 > d.nz)
                for (int l = 0; l < 64; ++l)
                    if (x0 + (l & 3) >= d.nx || y0 + ((l >> 2) & 3) >= d.ny || z0 + (l >> 4) >= d.nz) m |= 1ull << l;
        }
        /* a wave's 64 blocks are two words of bits */
        const unsigned long long bits = __ballot(w < n && m != 0ull);
        if (w < n) {
            L.occp[w] = m;
            if (L.occr) L.occr[w] = __builtin_bitreverse64(m);
            if ((threadIdx.x & 31u) == 0u) L.bitsp[w >> 5] = (uint32_t)(bits >> (threadIdx.x & 32u));
        }
    }
}

#define CODE_BYTES 8
/* Codes of the jump march: one workgroup per R x R rows of cells (R = 2^T, the
 * largest coded cube's edge) and 8 bytes of each row.  A row's bytes begin one
 * cell before the grid's, so a workgroup reads the cubes of one more R in x.
 * A cell is full when it has an occupied voxel or one outside the grid, or
 * lies outside the cell grid itself: no coded cube reaches past the grid.
 * Bound by the latency of its loads, which are independent (a thread per
 * cell): 8.4 us at 256^3, 24 at 512^3; a row of cells per workgroup, with the
 * loads of one y after the other, took 15 and 47. */
template <int T>
__global__ __launch_bounds__(256) void cell_codes_kernel(BrickDims d, const uint64_t* __restrict__ occp, uint32_t cg,
                                                         int32_t ncx, int32_t ncy, int32_t ncz, uint32_t ccx,
                                                         uint32_t ccy, uint8_t* __restrict__ codes)
{
    constexpr int R = 1 << T, H = R / 2, QB = CODE_BYTES, W = 4 * QB + R;
    __shared__ uint8_t full[R * R * W], pair[H * H * (W / 2)], top[W / R];
    const int32_t cy0 = (int32_t)blockIdx.x * R, cz0 = (int32_t)blockIdx.y * R, q0 = (int32_t)blockIdx.z * QB;
    const int32_t cx0 = 4 * q0 - R;
    const int32_t e = 1 << (cg - 2u);               /* 4x4x4 blocks per cell edge */
    const uint64_t px = (uint64_t)d.px, py = (uint64_t)d.py;
    for (int32_t i = threadIdx.x; i < R * R * W; i += blockDim.x) {
        const int32_t cx = cx0 + i % W, cy = cy0 + i / W % R, cz = cz0 + i / (W * R);
        const int32_t bx = cx * e, by = cy * e, bz = cz * e;
        bool occ = cx < 0 || cx >= ncx || cy >= ncy || cz >= ncz || bx + e > d.kx || by + e > d.ky || bz + e > d.kz;
        if (!occ) {
            uint64_t m = 0ull;
            for (int32_t z = bz; z < bz + e; ++z)
                for (int32_t y = by; y < by + e; ++y)
                    for (int32_t x = bx; x < bx + e; ++x)
                        m |= occp[(uint64_t)(x + 1) + px * ((uint64_t)(y + 1) + py * (uint64_t)(z + 1))];
            occ = m != 0ull;
        }
        full[i] = occ ? 1u : 0u;
    }
    for (int32_t i = threadIdx.x; i < W / R; i += blockDim.x) top[i] = 0u;
    __syncthreads();
    for (int32_t i = threadIdx.x; i < H * H * (W / 2); i += blockDim.x) {
        const int32_t x = i % (W / 2), y = i / (W / 2) % H, z = i / (W / 2 * H);
        const uint8_t* p = full + 2 * x + W * (2 * y + R * (2 * z));
        const uint32_t o = p[0] | p[1] | p[W] | p[W + 1] | p[W * R] | p[W * R + 1] | p[W * R + W] | p[W * R + W + 1];
        pair[i] = (uint8_t)o;
        if (o) top[x / H] = 1u;                     /* every writer writes 1 */
    }
    __syncthreads();
    const int32_t row_bytes = (int32_t)(ccx / 4u);
    for (int32_t i = threadIdx.x; i < R * R * QB; i += blockDim.x) {
        const int32_t q = q0 + i % QB, y = i / QB % R, z = i / (QB * R);
        if (q >= row_bytes || cy0 + y >= ncy || cz0 + z >= ncz) continue;
        uint32_t out = 0u;
        for (int k = 0; k < 4; ++k) {
            const int32_t x = 4 * q + k - 1 - cx0;
            const uint32_t c = full[x + W * (y + R * z)]                         ? 0u
                               : !top[x / R]                                     ? 3u
                               : !pair[x / 2 + W / 2 * (y / 2 + H * (z / 2))]    ? 2u
                                                                                 : 1u;
            out |= c << (2 * k);
        }
        codes[(uint64_t)q + (uint64_t)row_bytes * ((uint64_t)(cy0 + y + 1) + (uint64_t)ccy * (uint64_t)(cz0 + z + 1))] =
            (uint8_t)out;
    }
}

__global__ __launch_bounds__(256) void dense_from_bricks_kernel(BrickDims d, const uint8_t* __restrict__ bricks,
                                                                const int32_t* __restrict__ slot_off,
                                                                int32_t* __restrict__ dense)
{
    const int64_t n = (int64_t)d.nx * d.ny * d.nz;
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x) {
        const int32_t x = (int32_t)(i % d.nx);
        const int64_t r = i / d.nx;
        const int32_t y = (int32_t)(r % d.ny), z = (int32_t)(r / d.ny);
        dense[i] = slot_off[bricks[brick_byte(x, y, z)]];
    }
}

__global__ void fill_u8_kernel(uint8_t* p, uint64_t n, uint8_t v)
{
    const uint64_t n16 = n / 16;
    uint4 vv;
    const uint32_t w = (uint32_t)v * 0x01010101u;
    vv.x = vv.y = vv.z = vv.w = w;
    uint4* p16 = (uint4*)p;
    for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n16; i += (uint64_t)gridDim.x * blockDim.x)
        p16[i] = vv;
    for (uint64_t i = n16 * 16 + (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n;
         i += (uint64_t)gridDim.x * blockDim.x)
        p[i] = v;
}

__global__ void fill_u32_kernel(uint32_t* p, uint64_t n, uint32_t v)
{
    for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (uint64_t)gridDim.x * blockDim.x)
        p[i] = v;
}

__global__ __launch_bounds__(256) void copy_kernel(const uint4* __restrict__ src, uint4* __restrict__ dst, uint64_t n16)
{
    for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n16; i += (uint64_t)gridDim.x * blockDim.x)
        dst[i] = src[i];
}

/* 64 workgroups: 8 move 25 GB/s over the link, 32 to 128 all of its 50-53,
 * 512 less when a chunk is 2 MiB.  The host reuses a chunk between two of these
 * kernels without a barrier in the stream.  Loads and stores are therefore of
 * system scope: they see and leave nothing in the L2s, and the flag may be set
 * once all of them are done.  A 2 MiB chunk takes 39.5 us so; with plain
 * accesses between two system-scope fences 41.4 (fences of one wave a
 * workgroup) or 47 (of every wave), with an event after the kernel 45. */
#define CHUNK_COPY_BLOCKS 64
__global__ __launch_bounds__(256) void copy_chunk_kernel(const uint64_t* src, uint64_t* dst, uint32_t bytes,
                                                         uint32_t* count, uint32_t* flag, uint32_t seq)
{
    const uint32_t n = bytes / 8u, stride = gridDim.x * blockDim.x, first = blockIdx.x * blockDim.x + threadIdx.x;
    uint32_t i = first;
    for (; i + 3u * stride < n; i += 4u * stride) {
        uint64_t v[4];
#pragma unroll
        for (uint32_t k = 0; k < 4u; ++k) v[k] = load_system(src + i + k * stride);
#pragma unroll
        for (uint32_t k = 0; k < 4u; ++k) store_system(dst + i + k * stride, v[k]);
    }
    for (; i < n; i += stride) store_system(dst + i, load_system(src + i));
    if (first < (bytes & 7u)) store_system((uint8_t*)(dst + n) + first, load_system((const uint8_t*)(src + n) + first));
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");    /* this wave's stores are done */
    __syncthreads();
    if (threadIdx.x == 0 &&
        __hip_atomic_fetch_add(count, 1u, __ATOMIC_ACQ_REL, __HIP_MEMORY_SCOPE_AGENT) == gridDim.x - 1u) {
        __hip_atomic_store(count, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        __hip_atomic_store(flag, seq, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
    }
}

hipError_t launch_copy_chunk(const void* src, void* dst, size_t bytes, uint32_t* count, uint32_t* flag, uint32_t seq,
                             hipStream_t s)
{
    copy_chunk_kernel<<<CHUNK_COPY_BLOCKS, 256, 0, s>>>((const uint64_t*)src, (uint64_t*)dst, (uint32_t)bytes, count, flag,
                                                         seq);
    return hipGetLastError();
}

static unsigned grid_for(uint64_t n)
{
    uint64_t b = (n + 255) / 256;
    if (b > 65536u * 8u) b = 65536u * 8u;
    if (b < 1) b = 1;
    return (unsigned)b;
}

hipError_t launch_scan_offsets(const int32_t* dense, uint64_t n, int32_t lut_n, uint8_t* used, unsigned long long* bad,
                               hipStream_t s)
{
    const unsigned g = grid_for(n / 16u + 1u);    /* four int4 a thread */
    scan_offsets_kernel<<<g, 256, 0, s>>>(dense, n, lut_n, used, bad);
    return hipGetLastError();
}

hipError_t launch_check_emissive(const int32_t* emissive, int32_t n, uint64_t n_vox, const int32_t* offsets,
                                 const uint8_t* ids, const uint8_t* remap, uint32_t* bad, hipStream_t s)
{
    if (n <= 0) return hipSuccess;
    check_emissive_kernel<<<grid_for((uint64_t)n), 256, 0, s>>>(emissive, n, n_vox, offsets, ids, remap, bad);
    return hipGetLastError();
}

static unsigned blocks_grid(const BrickDims& d)
{
    return grid_for(d.n_padded);
}

hipError_t launch_blocks_from_bricks(const BrickDims& d, const uint8_t* bricks, const BlockLevels& L, hipStream_t s)
{
    blocks_kernel<0><<<blocks_grid(d), 256, 0, s>>>(d, nullptr, nullptr, const_cast<uint8_t*>(bricks), L);
    return hipGetLastError();
}

hipError_t launch_blocks_from_offsets(const BrickDims& d, const int32_t* dense, const uint8_t* lut, uint8_t* bricks,
                                      const BlockLevels& L, hipStream_t s)
{
    blocks_kernel<1><<<blocks_grid(d), 256, 0, s>>>(d, dense, lut, bricks, L);
    return hipGetLastError();
}

hipError_t launch_blocks_from_ids(const BrickDims& d, const uint8_t* dense, const uint8_t* remap, uint8_t* bricks,
                                  const BlockLevels& L, hipStream_t s)
{
    blocks_kernel<2><<<blocks_grid(d), 256, 0, s>>>(d, dense, remap, bricks, L);
    return hipGetLastError();
}

hipError_t launch_cell_codes(const BrickDims& d, const uint64_t* occp, const CellLayout& c, uint32_t* codes,
                             hipStream_t s)
{
    const int32_t e = 1 << c.shift;
    const int32_t nx = (d.nx + e - 1) / e, ny = (d.ny + e - 1) / e, nz = (d.nz + e - 1) / e;
    const uint32_t r = 1u << c.top;
    const dim3 grid(((uint32_t)ny + r - 1) / r, ((uint32_t)nz + r - 1) / r, (c.ex / 4u + CODE_BYTES - 1) / CODE_BYTES);
    if (c.top == 2u)
        cell_codes_kernel<2><<<grid, 256, 0, s>>>(d, occp, c.shift, nx, ny, nz, c.ex, c.ey, (uint8_t*)codes);
    else
        cell_codes_kernel<3><<<grid, 256, 0, s>>>(d, occp, c.shift, nx, ny, nz, c.ex, c.ey, (uint8_t*)codes);
    return hipGetLastError();
}

hipError_t launch_dense_from_bricks(const BrickDims& d, const uint8_t* bricks, const int32_t* slot_off, int32_t* dense,
                                    hipStream_t s)
{
    dense_from_bricks_kernel<<<grid_for((uint64_t)d.nx * d.ny * d.nz), 256, 0, s>>>(d, bricks, slot_off, dense);
    return hipGetLastError();
}

hipError_t launch_fill_u8(uint8_t* p, uint64_t n, uint8_t v, hipStream_t s)
{
    fill_u8_kernel<<<grid_for(n / 16 + 1), 256, 0, s>>>(p, n, v);
    return hipGetLastError();
}

hipError_t launch_copy(const void* src, void* dst, uint64_t bytes, hipStream_t s)
{
    const uint64_t n16 = bytes / 16;
    copy_kernel<<<grid_for(n16), 256, 0, s>>>((const uint4*)src, (uint4*)dst, n16);
    return hipGetLastError();
}

hipError_t launch_fill_u32(uint32_t* p, uint64_t n, uint32_t v, hipStream_t s)
{
    fill_u32_kernel<<<grid_for(n), 256, 0, s>>>(p, n, v);
    return hipGetLastError();
}

/* ---- voxelizer ---------------------------------------------------------------------------- */

/* int(float) with x86 cvttss2si semantics (non-finite or out of range ->
 * INT_MIN), the value the reference's llvmpipe path produces for the
 * z-range of degenerate triangles; sums wrap as 32-bit integers. */
__device__ __forceinline__ int32_t cvt_i32(float f)
{
    if (!(f >= -2147483648.0f && f < 2147483648.0f)) return INT32_MIN;
    return (int32_t)f;
}
__device__ __forceinline__ int32_t wrap_add(int32_t a, int32_t b) { return (int32_t)((uint32_t)a + (uint32_t)b); }

struct V2 { float x, y; };
__device__ __forceinline__ float dot2(V2 a, float bx, float by) { return a.x * bx + a.y * by; }
__device__ __forceinline__ bool finite3(f3 v)
{
    return vt_absf(v.x) < vt_inff() && vt_absf(v.y) < vt_inff() && vt_absf(v.z) < vt_inff();
}

/* Per-triangle state of voxelize.gs after the set-up (:55-208): the
 * swizzled vertices' edge functions in the three planes, the z-range plane
 * and the (x, y) bounds of the column loop. */
struct VoxTri {
    int32_t lut;                 /* swizzle: 0 (dominant x), 1 (dominant y), 2 (dominant z) */
    int32_t mn[3], mx[3];
    V2 nxy[3], nyz[3], nzx[3];
    float dxy[3], dyz[3], dzx[3];
    f3 np;
    float dMin, dMax, nzInv;
};

/* voxelize.vs:20-28 and the set-up of voxelize.gs; false for a triangle
 * with a non-finite vertex (skipped). */
__device__ __forceinline__ bool vox_setup(const VoxArgs& a, int64_t tri, VoxTri& T)
{
    const float rf[3] = { (float)a.d.nx, (float)a.d.ny, (float)a.d.nz };
    f3 v[3];
    bool finite = true;
#pragma unroll
    for (int k = 0; k < 3; ++k) {
        const float* p = a.verts + 3 * (size_t)a.idx[3 * tri + k];
        float ls[4];
        mat4_mul(a.M, p[0], p[1], p[2], 1.0f, ls);
        v[k] = mk(ls[0] * rf[0], ls[1] * rf[1], ls[2] * rf[2]);
        finite = finite && finite3(v[k]);
    }
    if (!finite) return false;
    f3 n = cross(v[1] - v[0], v[2] - v[1]);
    const float anx = vt_absf(n.x), any = vt_absf(n.y), anz = vt_absf(n.z);
    if (anx >= any && anx >= anz) {
#pragma unroll
        for (int k = 0; k < 3; ++k) v[k] = mk(v[k].y, v[k].z, v[k].x);
        n = mk(n.y, n.z, n.x);
        T.lut = 0;
    } else if (any >= anx && any >= anz) {
#pragma unroll
        for (int k = 0; k < 3; ++k) v[k] = mk(v[k].z, v[k].x, v[k].y);
        n = mk(n.z, n.x, n.y);
        T.lut = 1;
    } else {
        T.lut = 2;
    }
    const float amn[3] = { vt_minf(vt_minf(v[0].x, v[1].x), v[2].x), vt_minf(vt_minf(v[0].y, v[1].y), v[2].y),
                           vt_minf(vt_minf(v[0].z, v[1].z), v[2].z) };
    const float amx[3] = { vt_maxf(vt_maxf(v[0].x, v[1].x), v[2].x), vt_maxf(vt_maxf(v[0].y, v[1].y), v[2].y),
                           vt_maxf(vt_maxf(v[0].z, v[1].z), v[2].z) };
#pragma unroll
    for (int k = 0; k < 3; ++k) {
        T.mn[k] = (int32_t)vt_minf(vt_maxf(floorf(amn[k]), 0.0f), rf[k]);
        T.mx[k] = (int32_t)vt_minf(vt_maxf(ceilf(amx[k]), 0.0f), rf[k]);
    }
    const f3 ee[3] = { v[1] - v[0], v[2] - v[1], v[0] - v[2] };
#pragma unroll
    for (int k = 0; k < 3; ++k) {
        const f3 ek = ee[k];
        T.nxy[k] = (n.z >= 0.0f) ? V2{ -ek.y, ek.x } : V2{ ek.y, -ek.x };
        T.nyz[k] = (n.x >= 0.0f) ? V2{ -ek.z, ek.y } : V2{ ek.z, -ek.y };
        T.nzx[k] = (n.y >= 0.0f) ? V2{ -ek.x, ek.z } : V2{ ek.x, -ek.z };
        const f3 vk = v[k];
        if (a.mode == 0) {
            T.dxy[k] = dot2(T.nxy[k], 0.5f - vk.x, 0.5f - vk.y) +
                       0.5f * vt_maxf(vt_absf(T.nxy[k].x), vt_absf(T.nxy[k].y));
            T.dyz[k] = dot2(T.nyz[k], 0.5f - vk.y, 0.5f - vk.z) +
                       0.5f * vt_maxf(vt_absf(T.nyz[k].x), vt_absf(T.nyz[k].y));
            T.dzx[k] = dot2(T.nzx[k], 0.5f - vk.z, 0.5f - vk.x) +
                       0.5f * vt_maxf(vt_absf(T.nzx[k].x), vt_absf(T.nzx[k].y));
        } else {
            T.dxy[k] = (-dot2(T.nxy[k], vk.x, vk.y) + vt_maxf(0.0f, T.nxy[k].x)) + vt_maxf(0.0f, T.nxy[k].y);
            T.dyz[k] = (-dot2(T.nyz[k], vk.y, vk.z) + vt_maxf(0.0f, T.nyz[k].x)) + vt_maxf(0.0f, T.nyz[k].y);
            T.dzx[k] = (-dot2(T.nzx[k], vk.z, vk.x) + vt_maxf(0.0f, T.nzx[k].x)) + vt_maxf(0.0f, T.nzx[k].y);
        }
    }
    T.np = (n.z < 0.0f) ? -n : n;
    const float dTri = dot(T.np, v[0]);
    T.dMin = (a.mode == 0) ? dTri - (T.np.x * 0.5f + T.np.y * 0.5f)
                           : (dTri - vt_maxf(T.np.x, 0.0f)) - vt_maxf(T.np.y, 0.0f);
    T.dMax = (a.mode == 0) ? T.dMin : (dTri - vt_minf(T.np.x, 0.0f)) - vt_minf(T.np.y, 0.0f);
    T.nzInv = 1.0f / T.np.z;
    return true;
}

/* One (x, y) column of the triangle's loop (voxelize.gs:181-231): the 2D
 * edge test in the dominant plane, the z-range from the plane, the tests in
 * the other two planes, and the write of every covered voxel (unswizzled). */
__device__ __forceinline__ void vox_column(const VoxArgs& a, const VoxTri& T, int32_t x, int32_t y)
{
    const int32_t res[3] = { a.d.nx, a.d.ny, a.d.nz };
    const float fx = (float)x, fy = (float)y;
    const float d0 = T.dxy[0] + dot2(T.nxy[0], fx, fy);
    const float d1 = T.dxy[1] + dot2(T.nxy[1], fx, fy);
    const float d2 = T.dxy[2] + dot2(T.nxy[2], fx, fy);
    if (!(d0 >= 0.0f && d1 >= 0.0f && d2 >= 0.0f)) return;
    const float dnp = T.np.x * fx + T.np.y * fy;
    const float zMinInt = (-dnp + T.dMin) * T.nzInv;
    const float zMaxInt = (a.mode == 0) ? zMinInt : (-dnp + T.dMax) * T.nzInv;
    const float zMinFloor = floorf(zMinInt), zMaxCeil = ceilf(zMaxInt);
    int32_t zMin = wrap_add(cvt_i32(zMinFloor), -(int32_t)(zMinFloor == zMinInt));
    int32_t zMax = wrap_add(cvt_i32(zMaxCeil), (int32_t)(zMaxCeil == zMaxInt));
    if (zMin < T.mn[2]) zMin = T.mn[2];
    if (zMax > T.mx[2]) zMax = T.mx[2];
    for (int32_t z = zMin; z < zMax; ++z) {
        const float fz = (float)z;
        bool ok = true;
#pragma unroll
        for (int k = 0; k < 3; ++k) {
            ok = ok && (T.dyz[k] + dot2(T.nyz[k], fy, fz) >= 0.0f);
            ok = ok && (T.dzx[k] + dot2(T.nzx[k], fz, fx) >= 0.0f);
        }
        if (!ok) continue;
        int32_t c0, c1, c2;
        if (T.lut == 0) { c0 = z; c1 = x; c2 = y; }
        else if (T.lut == 1) { c0 = y; c1 = z; c2 = x; }
        else { c0 = x; c1 = y; c2 = z; }
        if ((uint32_t)c0 >= (uint32_t)res[0] || (uint32_t)c1 >= (uint32_t)res[1] || (uint32_t)c2 >= (uint32_t)res[2])
            continue;
        if (a.bricks) a.bricks[brick_byte(c0, c1, c2)] = a.slot;
        if (a.occ) a.occ[(size_t)c0 + (size_t)c1 * res[0] + (size_t)c2 * (size_t)res[0] * res[1]] = 1u;
    }
}

/* One thread per triangle.  Workgroup i works on triangle chunk
 * (i % 8) * per + i / 8: workgroups go to the eight XCDs in turn, so each
 * XCD takes one contiguous run of the triangle list (neighbouring triangles,
 * whose voxels share 64-byte lines, are then written from one L2 instead of
 * being merged from eight).  A triangle whose column loop exceeds
 * a.big_area columns is listed for voxelize_big_kernel instead. */
#define VOX_XCDS 8u
__global__ __launch_bounds__(256) void voxelize_kernel(VoxArgs a)
{
    const uint32_t per = (gridDim.x + VOX_XCDS - 1u) / VOX_XCDS;
    const uint64_t chunk = (uint64_t)(blockIdx.x % VOX_XCDS) * per + blockIdx.x / VOX_XCDS;
    const int64_t tri = (int64_t)chunk * blockDim.x + threadIdx.x;
    if (tri >= a.ntri) return;
    VoxTri T;
    if (!vox_setup(a, tri, T)) return;
    const int64_t w = T.mx[0] > T.mn[0] ? T.mx[0] - T.mn[0] : 0, h = T.mx[1] > T.mn[1] ? T.mx[1] - T.mn[1] : 0;
    if (a.big && w * h > a.big_area && tri < (int64_t)0xffffffff) {
        const uint32_t slot = atomicAdd(a.big_count, 1u);
        if (slot < a.big_cap) {
            a.big[slot] = (uint32_t)tri;
            return;
        }
    }
    for (int32_t x = T.mn[0]; x < T.mx[0]; ++x)
        for (int32_t y = T.mn[1]; y < T.mx[1]; ++y) vox_column(a, T, x, y);
}

/* The listed large triangles, one wave each: the lanes take the triangle's
 * (x, y) columns in turn (consecutive lanes, consecutive y). */
__global__ __launch_bounds__(256) void voxelize_big_kernel(VoxArgs a)
{
    const uint32_t lane = threadIdx.x & 63u;
    const uint32_t wave = blockIdx.x * (blockDim.x >> 6) + (threadIdx.x >> 6);
    const uint32_t waves = gridDim.x * (blockDim.x >> 6);
    const uint32_t n = *a.big_count < a.big_cap ? *a.big_count : a.big_cap;
    for (uint32_t i = wave; i < n; i += waves) {
        VoxTri T;
        if (!vox_setup(a, (int64_t)a.big[i], T)) continue;
        const int64_t w = T.mx[0] - T.mn[0], h = T.mx[1] - T.mn[1];
        for (int64_t k = lane; k < w * h; k += 64) vox_column(a, T, T.mn[0] + (int32_t)(k / h), T.mn[1] + (int32_t)(k % h));
    }
}

/* Bilinear quad table of an RGB image (EnvView::quad): one 64-byte entry per
 * (i0 + 1, j0 + 1) in [0, w] x [0, h], texels outside the image zero. */
__global__ __launch_bounds__(256) void env_quads_kernel(const float* __restrict__ img, int32_t w, int32_t h,
                                                        float4* __restrict__ quads)
{
    const uint64_t n = (uint64_t)(w + 1) * (uint64_t)(h + 1);
    for (uint64_t e = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; e < n; e += (uint64_t)gridDim.x * blockDim.x) {
        const int32_t i0 = (int32_t)(e % (uint64_t)(w + 1)) - 1, j0 = (int32_t)(e / (uint64_t)(w + 1)) - 1;
        float t[12];
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            const int32_t i = i0 + (k & 1), j = j0 + (k >> 1);
            const bool ok = i >= 0 && i < w && j >= 0 && j < h;
#pragma unroll
            for (int ch = 0; ch < 3; ++ch) t[3 * k + ch] = ok ? img[((size_t)j * w + i) * 3 + ch] : 0.0f;
        }
        float4* q = quads + e * 4u;
        q[0] = make_float4(t[0], t[1], t[2], t[3]);
        q[1] = make_float4(t[4], t[5], t[6], t[7]);
        q[2] = make_float4(t[8], t[9], t[10], t[11]);
        q[3] = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    }
}

hipError_t launch_env_quads(const float* img, int32_t w, int32_t h, float4* quads, hipStream_t s)
{
    const uint64_t n = (uint64_t)(w + 1) * (uint64_t)(h + 1);
    const uint64_t g = (n + 255) / 256;
    env_quads_kernel<<<(unsigned)(g < 65536 ? g : 65536), 256, 0, s>>>(img, w, h, quads);
    return hipGetLastError();
}

hipError_t launch_voxelize(const VoxArgs& a, int cus, hipStream_t s)
{
    if (a.ntri <= 0) return hipSuccess;
    /* a multiple of the XCD count, so the chunk mapping covers every chunk */
    const uint64_t g = (uint64_t)(a.ntri + 255) / 256;
    const uint64_t g8 = (g + VOX_XCDS - 1) / VOX_XCDS * VOX_XCDS;
    voxelize_kernel<<<(unsigned)g8, 256, 0, s>>>(a);
    if (a.big) {
        const uint64_t waves = (uint64_t)a.big_cap < (uint64_t)cus * 32u ? (uint64_t)a.big_cap : (uint64_t)cus * 32u;
        voxelize_big_kernel<<<(unsigned)((waves + 3) / 4), 256, 0, s>>>(a);
    }
    return hipGetLastError();
}

}  // namespace vt

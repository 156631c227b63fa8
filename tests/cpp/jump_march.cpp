/* The jump march's own source (vt_jump.h) on the CPU, one ray at a time:
 *   jump_march IN OUT
 * IN: int32 nx, ny, nz, n; float bmin[3], bmax[3]; the grid's voxels (a byte
 * each, x fastest); n rays as the queue holds them (float4, float2).
 * OUT: int32[4] a ray: 0 outside, 1 stopped or 2 stepwise, then the voxel.
 * The tables are exactly as long as the library's, so that the address
 * sanitizer finds every read outside them. */
#define VT_FN static inline
#include "vt_jump.h"
#include "vt_layout.h"

#include <cstdio>
#include <cstdlib>
#include <vector>

using namespace vt;

struct Tables {
    std::vector<uint64_t> masks;
    std::vector<uint32_t> codes;
};

static bool full(const std::vector<uint8_t>& v, const BrickDims& d, int x, int y, int z)
{
    if (x < 0 || y < 0 || z < 0 || x >= d.nx || y >= d.ny || z >= d.nz) return true;
    return v[(size_t)x + (size_t)d.nx * ((size_t)y + (size_t)d.ny * (size_t)z)] != 0;
}

/* Whether the aligned cube of cells holds only cells that lie whole in the
 * block grid and have no occupied voxel and none outside the grid. */
static Tables build(const std::vector<uint8_t>& v, const BrickDims& d, const CellLayout& c)
{
    Tables t;
    t.masks.assign((size_t)d.n_padded, ~0ull);
    for (int bz = 0; bz < d.kz; ++bz)
        for (int by = 0; by < d.ky; ++by)
            for (int bx = 0; bx < d.kx; ++bx) {
                uint64_t m = 0;
                for (int l = 0; l < 64; ++l)
                    if (full(v, d, 4 * bx + (l & 3), 4 * by + ((l >> 2) & 3), 4 * bz + (l >> 4))) m |= 1ull << l;
                t.masks[(size_t)(bx + 1) + (size_t)d.px * ((size_t)(by + 1) + (size_t)d.py * (size_t)(bz + 1))] = m;
            }
    const int e = 1 << c.shift;
    const int n[3] = { (d.nx + e - 1) / e, (d.ny + e - 1) / e, (d.nz + e - 1) / e };
    std::vector<uint8_t> occ((size_t)n[0] * n[1] * n[2]);
    for (int z = 0; z < n[2]; ++z)
        for (int y = 0; y < n[1]; ++y)
            for (int x = 0; x < n[0]; ++x) {
                bool o = false;
                for (int k = 0; k < e * e * e && !o; ++k)
                    o = full(v, d, x * e + k % e, y * e + k / e % e, z * e + k / (e * e));
                occ[(size_t)x + (size_t)n[0] * ((size_t)y + (size_t)n[1] * z)] = o;
            }
    auto any = [&](int x, int y, int z, int log) {
        const int r = 1 << log, x0 = x >> log << log, y0 = y >> log << log, z0 = z >> log << log;
        for (int k = z0; k < z0 + r; ++k)
            for (int j = y0; j < y0 + r; ++j)
                for (int i = x0; i < x0 + r; ++i)
                    if (i >= n[0] || j >= n[1] || k >= n[2] || occ[(size_t)i + (size_t)n[0] * ((size_t)j + (size_t)n[1] * k)]) return true;
        return false;
    };
    t.codes.assign(c.words, 0u);
    for (int z = 0; z < n[2]; ++z)
        for (int y = 0; y < n[1]; ++y)
            for (int x = 0; x < n[0]; ++x) {
                const uint32_t code = any(x, y, z, 0) ? 0u : !any(x, y, z, (int)c.top) ? 3u : !any(x, y, z, 1) ? 2u : 1u;
                const size_t i = (size_t)(x + 1) + (size_t)c.ex * ((size_t)(y + 1) + (size_t)c.ey * (size_t)(z + 1));
                t.codes[i >> 4] |= code << (2 * (i & 15));
            }
    return t;
}

/* The loop of wf_traverse_kernel for one lane. */
template <bool FINE>
static bool trace(JumpState& J, const GridView& g, int limit)
{
    for (int k = 0; k < limit; ++k) {
        bool live = true;
        int32_t edge = 0;
        jump_march<FINE, false>(J, g, 32, 1, live, edge);
        if (live) continue;
        if (edge < 0) return true;
        const int32_t x = J.x, y = J.y, z = J.z;
        if (!J.near_jump<false>(g, edge)) J.resolve(g, edge);
        if (J.x < x || J.y < y || J.z < z || (J.x == x && J.y == y && J.z == z)) return false;
    }
    return false;
}

int main(int argc, char** argv)
{
    if (argc < 3) return 2;
    FILE* f = fopen(argv[1], "rb");
    int32_t h[4];
    float b[6];
    if (!f || fread(h, 4, 4, f) != 4 || fread(b, 4, 6, f) != 6) return 2;
    std::vector<uint8_t> v((size_t)h[0] * h[1] * h[2]);
    std::vector<float> rays((size_t)h[3] * 6);
    if (fread(v.data(), 1, v.size(), f) != v.size() || fread(rays.data(), 4, rays.size(), f) != rays.size()) return 2;
    fclose(f);
    const BrickDims d = make_dims(h[0], h[1], h[2]);
    const CellLayout c = cell_layout(d);
    const Tables t = build(v, d, c);
    GridView g = {};
    g.nx = d.nx; g.ny = d.ny; g.nz = d.nz;
    g.rx = (float)d.nx; g.ry = (float)d.ny; g.rz = (float)d.nz;
    for (int k = 0; k < 3; ++k) { g.bmin[k] = b[k]; g.bmax[k] = b[3 + k]; g.ext[k] = 1.0f / (b[3 + k] - b[k]); }
    g.bxp = (uint32_t)d.px; g.byp = (uint32_t)d.py;
    g.occp = t.masks.data();
    g.codes = t.codes.data();
    g.code_words = c.words;
    g.ccx = c.ex; g.ccy = c.ey; g.cg = c.shift; g.cedge = c.edges();
    g.jc0 = jump_bound0(std::max(d.nx, std::max(d.ny, d.nz)));
    std::vector<int32_t> out((size_t)h[3] * 4);
    for (int i = 0; i < h[3]; ++i) {
        const float* r = &rays[(size_t)i * 6];
        JumpState J;
        const int st = J.init(g, { r[0], r[1], r[2], r[3] }, { r[4], r[5] });
        int32_t* o = &out[(size_t)i * 4];
        o[0] = st;
        if (st != JumpState::READY) continue;
        const int limit = d.nx + d.ny + d.nz + 8;
        if (!(c.shift == 2 ? trace<true>(J, g, limit) : trace<false>(J, g, limit))) o[0] = -1;
        o[1] = J.gx(); o[2] = J.gy(); o[3] = J.gz();
    }
    f = fopen(argv[2], "wb");
    if (!f || fwrite(out.data(), 4, out.size(), f) != out.size()) return 2;
    fclose(f);
    return 0;
}

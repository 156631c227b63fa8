/*
 * vt_kernels.h - kernel argument blocks and launchers shared by the HIP
 * translation units of the voxel path tracer.
 */
#pragma once

#include "vt_device.h"
#include "vt_layout.h"

namespace vt {

struct TraceArgs {
    GridView g;
    EnvView e;
    CamView c;
    Settings s;
    const MatRec* recs;          /* 256 records: [0] = offset 0 (ground), [slot] */
    int32_t W, H;
    uint64_t seed;
    uint32_t n0, count, rng_frame_max;
    float4* accum;
    double* sum64;
    unsigned long long* stats;   /* 6 counters */
    uint32_t* tile_counter;
    int32_t tiles_x, n_tiles;
    int32_t lds_bits;            /* stage occupancy bits in LDS */
    int32_t step;                /* wavefront traversal marches step by step (step_march) */
    int32_t lds_bits_p;          /* step-by-step wavefront traversal: stage the padded block bits in LDS */
    int32_t cdfv_lds_bytes;
    int32_t dda_budget;          /* wavefront traversal: jumps or DDA steps between refill checks */
    int32_t refill_min;          /* wavefront traversal: idle lanes that trigger a refill */
    int32_t refill_chunk;        /* wavefront traversal: queue entries dealt to a workgroup at a time */
};

struct Counters {
    uint32_t rays, visits, interactions, samples, env_samples, env_evals;
};

enum { PH_PRIMARY = 0, PH_SHADOW = 1, PH_CONT = 2, PH_COMB = 3 /* shade round: shadow result, then CONT */ };

/* Registers of one path between traversals. */
struct PathState {
    f3 ray_o, ray_d;             /* the ray to trace next */
    f3 basis_o;                  /* origin voxelSpaceToWorldSpace re-intersects from */
    f3 throughput, radiance;
    f3 direct;                   /* light-sample contribution pending its shadow ray */
    f3 factor;                   /* f * |cos| / pdf of the sampled continuation */
    f3 next_d;                   /* continuation direction */
    float bsdf_pdf;
    int32_t ex, ey, ez;          /* emissive voxel the shadow ray must reach */
    int32_t light_is_voxel;
    int32_t phase, bounces;
    vt_pcg32 rng;
};

/* Wavefront path storage: one slot per path of a chunk of the launch's
 * (pass, pixel) space, structure-of-arrays in HBM. */
/* Path state by queue position: the fields of the path whose ray sits at
 * position j of a ray queue are at index j of that queue's buffer, so shade
 * kernels read and write them contiguously (a surviving path moves to its
 * position in the next queue). */
struct PathBuf {
    float4* o;        /* ray_o (or basis origin after generate).xyz, bsdf_pdf */
    float4* nd;       /* continuation direction (camera direction after generate), pixel (bits) */
    float4* thr;      /* throughput times the continuation factor, sample slot of the chunk (bits) */
    float4* rad;      /* radiance if the light sample is occluded, emissive target x | y << 16 (bits) */
    float4* dir;      /* radiance if it is visible, target z | light_is_voxel << 15 | bounces << 16 (bits) */
    float4* fac;      /* batch and cache launches only: w = scene or training slot + 1 (bits) */
    uint4* meta;      /* after generate only: pixel, sample slot, bounces (0), scene or training slot + 1 */
    uint64_t* rng;    /* PCG32 state (increment = 2*pixel+1) */
};

/* Traversal result in 8 bytes: voxel coordinates + 1 (they lie in [-1, n]
 * for n <= 4096) in 16-bit fields, kind in the top half of the second word. */
__device__ __forceinline__ uint2 pack_hit(int32_t x, int32_t y, int32_t z, int32_t kind)
{
    return make_uint2((uint32_t)(x + 1) | ((uint32_t)(y + 1) << 16), (uint32_t)(z + 1) | ((uint32_t)kind << 16));
}
__device__ __forceinline__ int32_t unpack_hit(uint2 r, Hit& h)
{
    h.x = (int32_t)(r.x & 0xffffu) - 1;
    h.y = (int32_t)(r.x >> 16) - 1;
    h.z = (int32_t)(r.y & 0xffffu) - 1;
    return (int32_t)(r.y >> 16);
}

/* A queue of paths has QUEUE_PARTS parts with a length of their own, in lines
 * of their own: a length that workgroups of all XCDs add to takes 13 ns an
 * addition, which bound the kernels that append (65 k additions a launch).  The
 * positions of the parts are interleaved by runs of QUEUE_RUN paths, so a part
 * needs no share of the arrays of its own; part s holds its m-th path at
 * queue_position(s, m).  Work units of one size (threads of a workgroup) append
 * to parts in turn (queue_part), every 16 units in another order, so that a
 * pattern of the image does not fill one part more than another.  Positions up
 * to the longest part's end are visited, those past a part's length are empty. */
enum : uint32_t { QUEUE_PARTS = 16, QUEUE_RUN = 64, QUEUE_COUNT_STRIDE = 32 };
__host__ __device__ inline uint32_t queue_position(uint32_t s, uint32_t m)
{
    return (m / QUEUE_RUN * QUEUE_PARTS + s) * QUEUE_RUN + m % QUEUE_RUN;
}
__host__ __device__ inline uint32_t queue_part(uint32_t unit)
{
    return (unit + ((unit / QUEUE_PARTS * 0x9e3779b1u) >> 28)) % QUEUE_PARTS;
}
/* Positions that a chunk of `paths` paths needs in any round, for units of at
 * most 1024 paths: QUEUE_PARTS units that are full, rounded up to the next run
 * of rounds' units (queue_part gives each part one of QUEUE_PARTS units). */
inline uint64_t queue_positions(uint64_t paths)
{
    return (paths + QUEUE_PARTS * 1024u - 1u) / (QUEUE_PARTS * 1024u) * (QUEUE_PARTS * 1024u);
}

/* LDS of a traversal workgroup after its table: the list counter and the
 * lengths of the queue's parts. */
enum : uint32_t { WF_TAKEN_BYTES = 16 + QUEUE_PARTS * 4 };

struct WfPaths {
    PathBuf s[2];     /* state of the paths in queue 0 / queue 1 */
    uint2* hit;       /* traversal result per queue entry (pack_hit): x, y, z (each + 1), kind */
    float4* smp;      /* finished tonemapped sample of each path of the chunk */
    float4* qa0;      /* ray queue 0 (2 x cap entries: a path's shadow and continuation rays at 2k, 2k + 1):
                         origin.xyz moved by sign(d)*0.001, 1/clamped d.x */
    float2* qb0;      /*              1/clamped d.y, 1/clamped d.z */
    uint32_t* qt0;    /*              scene of the ray (batch launches only) */
    float4* qa1;      /* ray queue 1 */
    float2* qb1;
    uint32_t* qt1;
    uint32_t* cnt;    /* paths in each part of queue 0, then of queue 1 (queue_count) */
    uint64_t cap;     /* slots */
};

/* A batch of scenes rendered by one wavefront launch: per-scene arguments
 * and the prefix sums of their path counts (W*H*count) and pixel counts
 * (W*H), n + 1 entries each. */
struct BatchTable {
    const TraceArgs* tab;
    const uint64_t* path_base;
    const uint64_t* pix_base;
    uint32_t n;
    unsigned long long* stats;   /* 6 counters or null */
    int32_t packed;              /* every scene has packed-march masks (GridView::occr) */
    int32_t step;                /* a scene marches step by step, so all do */
};

/* Radiance-cache rendering of one pass: paths that are not training paths
 * end into the cache at their vertex of bounce cache_bounce (query appended
 * to q_*); training paths (path index % train_stride == train_offset, slot =
 * index / train_stride) run the plain integrator and record each shaded
 * vertex (query, throughput, radiance so far: 18 floats), and when they end
 * append one training sample per vertex: target = (R_end - R_v) / T_v. */
struct CacheRender {
    int32_t cache_bounce;   /* bounce at which paths end into the cache (-1 never) */
    int32_t train_bounce;   /* the same for training paths */
    uint32_t train_stride, train_offset, train_slots, max_vertices;
    float* vrec;            /* [train_slots][max_vertices][18] */
    uint32_t* vrec_n;       /* [train_slots] */
    float* q_raw;           /* [paths][12] */
    uint4* q_meta;          /* [paths] metadata of the path that ended into the cache */
    float4* q_rad;          /* [paths] its radiance and throughput at that point */
    float4* q_thr;
    float* q_out;           /* [paths][3] */
    uint32_t* q_count;
    uint32_t* q_done;       /* queries already answered */
    float* s_raw;           /* [s_cap][12] */
    float* s_tgt;           /* [s_cap][3] */
    uint32_t* s_count;
    uint32_t s_cap;
};

size_t render_lds_bytes(const TraceArgs& a);
/* One pass (a.count must be 1) of cache rendering into a.accum. */
hipError_t launch_render_cached(const TraceArgs& a, const WfPaths& P, const CacheRender& C, const void* pack,
                                const float* bias, int cus, hipStream_t s);
/* Wavefront render of every scene of B (paths of all scenes share the
 * queues; rounds follow the largest max_bounces, paths of scenes with fewer
 * bounces finish earlier).  a0 supplies the traversal tuning. */
hipError_t launch_render_batch(const TraceArgs& a0, const BatchTable& B, const WfPaths& P, uint64_t total_paths,
                               uint64_t total_pixels, int max_bounces, int cus, hipStream_t s, bool stats);
/* Events recorded on the launch stream around traversal launches: pair k
 * brackets the k-th timed launch (at most cap pairs; *used counts them). */
struct LaunchTimer {
    hipEvent_t* ev;
    int cap;
    int* used;
};

/* Wavefront render of the launch in a: path chunks of at most P.cap slots,
 * 1 + max_bounces traverse/shade rounds per chunk (each round after the
 * first traces a shadow and a continuation ray per path).  With acc_wait, every
 * accumulation launch first waits for that event (passes accumulate in
 * order when two launches render consecutive passes on two streams). */
hipError_t launch_render_wavefront(const TraceArgs& a, const WfPaths& P, int cus, hipStream_t s, bool stats,
                                   const LaunchTimer* timer = nullptr, hipEvent_t acc_wait = nullptr);
hipError_t launch_render(const TraceArgs& a, int grid, hipStream_t s, bool stats);
int render_blocks_per_cu(const TraceArgs& a, bool stats);
/* The jump march of a single grid reads its codes from LDS address 0, where a
 * kernel's dynamic LDS begins if it has no other: an error if one has. */
hipError_t check_lds_base();
hipError_t launch_first_hit(const TraceArgs& a, int32_t* out, hipStream_t s);
hipError_t launch_trace_rays(const TraceArgs& a, int32_t n, const float* o, const float* d, int32_t* out,
                             uint32_t* count, uint32_t* flag, uint32_t seq, hipStream_t s);
hipError_t launch_reset_counter(uint32_t* c, unsigned long long* stats, hipStream_t s);
/* The same, and the megakernel's block bits (GridView::bits) unless null. */
hipError_t launch_render_setup(const GridView& g, uint32_t* bits, uint32_t* c, unsigned long long* stats, hipStream_t s);
hipError_t launch_device_math(int32_t fn, int32_t n, const float* a, const float* b, float* out, hipStream_t s);

/* ---- volume layout (BrickDims: vt_layout.h) --------------------------------------------- */
/* Which material offsets a dense int32 grid uses: used[o] = 1 for every o in
 * [0, lut_n) that occurs (used zero at launch); *bad = the smallest index of
 * an offset >= lut_n (all ones at launch). */
hipError_t launch_scan_offsets(const int32_t* dense, uint64_t n, int32_t lut_n, uint8_t* used, unsigned long long* bad,
                               hipStream_t s);
/* *bad = the smallest i whose emissive[i] lies outside [0, n_vox) or is an
 * empty voxel of the dense grid (offsets, or ids with their remap; the other
 * null); all ones at launch. */
hipError_t launch_check_emissive(const int32_t* emissive, int32_t n, uint64_t n_vox, const int32_t* offsets,
                                 const uint8_t* ids, const uint8_t* remap, uint32_t* bad, hipStream_t s);
/* The block levels (GridView: masks occp, their bit-reversed copy occr unless
 * null, bits bitsp) of the padded block grid.  From the bricks, or from a
 * dense grid (offsets with lut, or ids with remap), which also writes the
 * bricks. */
struct BlockLevels {
    uint64_t* occp;
    uint64_t* occr;
    uint32_t* bitsp;
};
hipError_t launch_blocks_from_bricks(const BrickDims& d, const uint8_t* bricks, const BlockLevels& L, hipStream_t s);
hipError_t launch_blocks_from_offsets(const BrickDims& d, const int32_t* dense, const uint8_t* lut, uint8_t* bricks,
                                      const BlockLevels& L, hipStream_t s);
hipError_t launch_blocks_from_ids(const BrickDims& d, const uint8_t* dense, const uint8_t* remap, uint8_t* bricks,
                                  const BlockLevels& L, hipStream_t s);
/* The jump march's codes (GridView::codes) from the padded masks.  The largest
 * coded cube has 2^top cells an edge (top 2 or 3), the next 2, the smallest 1.
 * The codes of the padding are not written (zero). */
hipError_t launch_cell_codes(const BrickDims& d, const uint64_t* occp, const CellLayout& c, uint32_t* codes,
                             hipStream_t s);
/* Bricked slots -> dense int32 offsets via slot_off[256]. */
hipError_t launch_dense_from_bricks(const BrickDims& d, const uint8_t* bricks, const int32_t* slot_off, int32_t* dense,
                                    hipStream_t s);
/* Fill a byte buffer (graph-safe replacement for hipMemsetAsync). */
hipError_t launch_fill_u8(uint8_t* p, uint64_t n, uint8_t v, hipStream_t s);
/* Emissive list -> (x, y, z, slot) per entry, from the current grid. */
hipError_t launch_light_table(const GridView& g, int4* out, hipStream_t s);
hipError_t launch_env_quads(const float* img, int32_t w, int32_t h, float4* quads, hipStream_t s);
hipError_t launch_fill_u32(uint32_t* p, uint64_t n, uint32_t v, hipStream_t s);
/* Streaming 16-byte-vector copy (bytes must be a multiple of 16). */
hipError_t launch_copy(const void* src, void* dst, uint64_t bytes, hipStream_t s);

/* ---- voxelizer ------------------------------------------------------------------------- */
struct VoxArgs {
    BrickDims d;
    const float* verts;
    const uint32_t* idx;
    int64_t ntri;
    float M[16];
    int32_t mode;                /* 0 THIN, 1 FAT */
    uint8_t slot;
    uint8_t* bricks;             /* may be null */
    uint8_t* occ;                /* dense occupancy, may be null */
    /* triangles with more than big_area (x, y) columns go to a list of
     * big_cap entries (counter big_count, zero at launch) that one wave per
     * triangle then voxelizes; big = null keeps every triangle on one thread */
    uint32_t* big;
    uint32_t* big_count;
    uint32_t big_cap;
    int32_t big_area;
};
hipError_t launch_voxelize(const VoxArgs& a, int cus, hipStream_t s);

}  // namespace vt

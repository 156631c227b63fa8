"""The jump march (renders without statistics) against the step-by-step march
(renders with statistics, bit-exact with the oracle) and the oracle itself: at
the sizes where the cells, the coded cubes and the padding change."""
import math

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def bits_equal(a, b):
    return ((a.view(np.uint32) == b.view(np.uint32)) | (np.isnan(a) & np.isnan(b))).all()


def scene_of(shape, rng, fill=0.0005):
    """A floor of varying height, loose voxels, an emitter and a metal."""
    from voxeltoy_amd import api, scenes
    nz, ny, nx = shape
    recs = [scenes.lambert((0, 0, 0), (0.6, 0.55, 0.5)), scenes.lambert((5.0, 4.0, 3.0), (0.5, 0.5, 0.5)),
            scenes.metal((0, 0, 0), (0.9, 0.85, 0.8), 0.3)]
    mat, offs = scenes.build_materials(recs)
    id_offset = np.full(256, -1, np.int32)
    id_offset[1:4] = offs
    ids = np.zeros(shape, np.uint8)
    h = rng.integers(0, max(1, ny // 8) + 1, (nz // 8 + 1, nx // 8 + 1)).repeat(8, 0).repeat(8, 1)[:nz, :nx]
    for y in range(int(h.max())):
        ids[:, y, :][h > y] = 1
    n = max(3, int(fill * ids.size))
    at = rng.integers(0, ids.size, min(n, 200000))
    ids.reshape(-1)[at] = rng.choice(np.array([1, 2, 3], np.uint8), len(at), p=[0.6, 0.2, 0.2])
    sc = scenes.Scene(ids, id_offset, mat)
    em = np.sort(at[ids.reshape(-1)[at] == 2])[:4096].astype(np.int32)
    sc.emissive = np.unique(em)
    return sc


def workload_of(shape, lens, width, height, rng):
    from voxeltoy_amd import scenes, workloads
    sc = scene_of(shape, rng)
    bmin, bmax = workloads.reference_bounds(sc.shape)
    cam = scenes.orbit_camera(bmin, bmax, math.radians(112), math.radians(float(rng.uniform(0, 360))), width, height,
                              lens_model=lens, lens_radius=4.0, focal_distance=900.0)
    return workloads.Workload("jump", sc, cam, width, height, spp=2, bounces=4, bmin=bmin, bmax=bmax,
                              env_top=(1.5, 1.4, 1.2), env_bottom=(0.3, 0.3, 0.35))


# cells of 4 voxels with cubes of up to 4 and 8 cells (57 cells an axis on), extents around multiples of 4,
# 16 and 32; cells of 8 (too many of 4 for the LDS); one cell; slabs
@pytest.mark.parametrize("shape,lens", [((4, 4, 4), 0), ((5, 3, 9), 1), ((33, 31, 32), 0), ((64, 17, 65), 2),
                                        ((21, 45, 224), 1), ((37, 16, 229), 0), ((256, 40, 255), 2),
                                        ((1, 64, 64), 0), ((264, 264, 266), 0), ((272, 270, 275), 1), ((6, 7, 4096), 0)])
def test_jump_march_equals_step_by_step(ctx, shape, lens):
    from voxeltoy_amd import workloads
    rng = np.random.default_rng(sum(shape) + lens)
    wl = workload_of(shape, lens, 333, 251, rng)
    workloads.load(ctx, wl)
    ctx.set_stats(True)
    ctx.render(wl.seed, 0, wl.spp)
    want = ctx.read_accum()
    ctx.set_stats(False)
    ctx.reset_accum()
    ctx.render(wl.seed, 0, wl.spp)
    assert bits_equal(ctx.read_accum(), want)


@pytest.mark.parametrize("shape", [(24, 20, 28), (18, 11, 240)])
def test_jump_march_equals_oracle(ctx, orc, shape):
    from voxeltoy_amd import workloads
    wl = workload_of(shape, 0, 96, 64, np.random.default_rng(shape[2]))
    workloads.load(ctx, wl)
    ctx.render(wl.seed, 0, wl.spp)
    sc = wl.scene
    o = orc.OracleScene(sc.offsets(), sc.mat, sc.emissive)
    o.set_camera(**wl.camera_arrays())
    o.set_environment(wl.env_top, wl.env_bottom)
    o.set_settings(max_bounces=wl.bounces)
    ref, _ = o.render(wl.width, wl.height, wl.seed, 0, wl.spp)
    assert bits_equal(ctx.read_accum(), ref)


def test_jump_march_in_cells_of_16(ctx):
    """A grid whose cells of 8 voxels are too many for the LDS, alone and in a
    batch with a small one (per-lane grids)."""
    from voxeltoy_amd import api, workloads
    rng = np.random.default_rng(9)
    big = workload_of((560, 552, 548), 0, 320, 200, rng)
    small = workload_of((30, 40, 50), 1, 120, 90, rng)
    workloads.load(ctx, big)
    ctx.set_stats(True)
    ctx.render(big.seed, 0, big.spp)
    want = ctx.read_accum()
    ctx.set_stats(False)
    ctx.reset_accum()
    ctx.render(big.seed, 0, big.spp)
    assert bits_equal(ctx.read_accum(), want)
    ctx.reset_accum()
    with api.Context(0) as other:
        workloads.load(other, small)
        other.set_stats(True)
        other.render(small.seed, 0, small.spp)
        want_small = other.read_accum()
        other.set_stats(False)
        other.reset_accum()
        b = api.Batch([ctx, other])
        b.render([big.seed, small.seed], [big.spp, small.spp])
        assert bits_equal(ctx.read_accum(), want)
        assert bits_equal(other.read_accum(), want_small)
        b.close()


def test_jump_march_full_shading_scene(ctx):
    """The 256^3 full-shading scene, 1.4 M camera rays: the statistics render
    and the plain one are the same image."""
    from voxeltoy_amd import workloads
    wl = workloads.full(1201, 583, spp=2)
    workloads.load(ctx, wl)
    ctx.set_stats(True)
    ctx.render(wl.seed, 0, wl.spp)
    want = ctx.read_accum()
    ctx.set_stats(False)
    ctx.reset_accum()
    ctx.render(wl.seed, 0, wl.spp)
    assert bits_equal(ctx.read_accum(), want)

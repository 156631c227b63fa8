"""Material records of the slots in use: edits, more and fewer slots, a slot that
the voxelizer adds, against the oracle."""
import numpy as np
import pytest

from test_gpu_jump_march import bits_equal

pytestmark = pytest.mark.gpu


def test_records_follow_the_materials(ctx, orc):
    from voxeltoy_amd import api, scenes, workloads
    rng = np.random.default_rng(4)
    shape = (20, 14, 22)
    bmin, bmax = workloads.reference_bounds(shape)
    cam = scenes.orbit_camera(bmin, bmax, 2.0, 0.7, 65, 47)

    def check(off, mat):
        wl = workloads.Workload("m", None, cam, 65, 47, spp=2, bounces=3, bmin=bmin, bmax=bmax)
        ctx.reset_accum()
        ctx.render(9, 0, 2)
        o = orc.OracleScene(off, mat)
        o.set_camera(**wl.camera_arrays())
        o.set_environment((1.5, 1.4, 1.2), (0.3, 0.3, 0.35))
        o.set_settings(max_bounces=3)
        ref, _ = o.render(65, 47, 9, 0, 2)
        assert bits_equal(ctx.read_accum(), ref)

    first = True
    for n in (3, 255, 1, 40):
        recs = [scenes.lambert((0, 0, 0), rng.uniform(0.2, 0.9, 3)) if k % 3 else scenes.metal((0, 0, 0), rng.uniform(0.5, 0.9, 3), 0.3)
                for k in range(n + 1)]
        mat, offs = scenes.build_materials(recs)
        mat = np.asarray(mat, np.float32)
        off = np.where(rng.random(shape) < 0.2, np.asarray(offs, np.int32)[rng.integers(0, n, shape)], -1).astype(np.int32)
        ctx.set_volume(off, mat)
        if first:
            wl = workloads.Workload("m", None, cam, 65, 47, spp=2, bounces=3, bmin=bmin, bmax=bmax)
            ctx.set_camera(**wl.camera_arrays())
            ctx.set_environment(top=(1.5, 1.4, 1.2), bottom=(0.3, 0.3, 0.35))
            ctx.set_settings(max_bounces=3)
            ctx.set_frame(65, 47)
            first = False
        check(off, mat)
        for k in (0, n // 2, n - 1):
            mat[offs[k] + 4:offs[k] + 7] = rng.uniform(0.1, 0.9, 3)
            ctx.update_material(int(offs[k]) + 4, mat[offs[k] + 4:offs[k] + 7])
        check(off, mat)
        if n < 255:
            # a material that no voxel had
            v = np.array([[-0.6, -0.5, 0.1], [0.7, -0.4, 0.2], [0.0, 0.6, -0.3]], np.float32)
            M = api.mesh_transform(v.min(0), v.max(0), shape[::-1])
            occ = ctx.voxelize(v, np.array([[0, 1, 2]], np.uint32), M, material_offset=int(offs[n]))
            off = np.where(occ != 0, np.int32(offs[n]), off)
            check(off, mat)

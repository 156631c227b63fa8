"""Picking rays through the codes of empty cubes and the pinned staging memory, against the oracle's step-by-step
march: whole and partial waves, the last staged size and the first unstaged one, cells of 4 and 8 voxels."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape,n", [((1, 1, 1), 1), ((5, 3, 9), 63), ((33, 31, 70), 64), ((126, 20, 126), 65),
                                     ((64, 57, 229), 16384), ((64, 57, 229), 16385), ((272, 270, 275), 4001)])
def test_records_equal_oracle(ctx, orc, shape, n):
    rng = np.random.default_rng(n)
    off = np.where(rng.random(shape) < min(0.3, 300.0 / np.prod(shape) ** 0.75), 0, -1).astype(np.int32)
    off.reshape(-1)[-1] = 0
    mat = np.array([0, 0, 0, 0, .5, .5, .5, 0], np.float32)
    ctx.set_volume(off, mat)
    o_sc = orc.OracleScene(off, mat)
    bmin, bmax, _ = ctx.bounds()
    o = (bmin + rng.uniform(-0.05, 1.05, (n, 3)) * (bmax - bmin)).astype(np.float32)
    d = rng.standard_normal((n, 3))
    d[: n // 4, rng.integers(0, 3)] = 0.0                # along a face, and along an edge
    d[: n // 16, :2] = 0.0
    d = (d / np.maximum(np.linalg.norm(d, axis=1, keepdims=True), 1e-30)).astype(np.float32)
    d[::97] = np.sign(d[::97])                           # axes that step together
    want = o_sc.trace_rays(o, d)
    assert np.array_equal(ctx.trace_rays(o, d), want)
    if n <= 16384:
        assert np.array_equal(ctx.trace_rays_noalloc(o, d), want)

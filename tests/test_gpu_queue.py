"""Renders whose path queues fill the parts of a queue unevenly (fewer paths than a unit, than a run, than the parts
hold) or in several chunks, against the one-kernel renderer, which has no queues."""
import numpy as np
import pytest

from test_gpu_jump_march import workload_of

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("width,height,chunk", [(1, 1, 0), (8, 8, 0), (33, 31, 0), (32, 32, 0), (205, 5, 0),
                                                (128, 128, 0), (129, 127, 4096), (257, 129, 16385)])
def test_queues_equal_one_kernel(ctx, width, height, chunk):
    from voxeltoy_amd import workloads
    rng = np.random.default_rng(width)
    wl = workload_of((33, 31, 46), 0, width, height, rng)
    workloads.load(ctx, wl)
    try:
        ctx.set_render_mode(0)
        ctx.render(wl.seed, 0, 3)
        want = ctx.read_accum()
        ctx.reset_accum()
        ctx.set_render_mode(1, chunk)
        ctx.render(wl.seed, 0, 3)
        got = ctx.read_accum()
    finally:
        ctx.set_render_mode(1)
    assert np.array_equal(got.view(np.uint32), want.view(np.uint32))

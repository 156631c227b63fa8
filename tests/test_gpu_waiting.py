"""Calls behind a long render: what they cost the host and other contexts."""
import time

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def long_render(ctx, seconds=0.5):
    """Loads the full-shading scene and starts a render of about `seconds`."""
    from voxeltoy_amd import workloads
    wl = workloads.full(1024, 1024, spp=1)
    workloads.load(ctx, wl)
    ctx.render(wl.seed, 0, 16)
    ctx.synchronize()
    t = time.perf_counter()
    ctx.render(wl.seed, 16, 32)
    ctx.synchronize()
    each = (time.perf_counter() - t) / 32
    ctx.render(wl.seed, 48, int(seconds / each) + 1)


def test_readback_behind_a_render_leaves_the_cores_idle(ctx):
    long_render(ctx)
    wall, cpu = time.perf_counter(), time.process_time()
    img = ctx.read_accum()
    wall, cpu = time.perf_counter() - wall, time.process_time() - cpu
    assert np.isfinite(img[..., 3]).all()
    assert wall > 0.2
    assert cpu < 1.8 * wall, (cpu, wall)      # the caller, if the runtime's wait spins; not four threads

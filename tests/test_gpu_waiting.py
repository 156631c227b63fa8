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


def test_pick_behind_a_render_holds_up_no_other_context(ctx, vtapi):
    """vt_trace_rays on a context whose render goes on, and meanwhile a pick
    through vt_trace_rays_noalloc on another context."""
    import threading
    from voxeltoy_amd import workloads
    o = np.array([[0.0, 400.0, 0.0]], np.float32)
    d = np.array([[0.1, -0.99, 0.1]], np.float32)
    with vtapi.Context(0) as other:
        workloads.load(other, workloads.small(1))
        want = other.trace_rays(o, d)
        long_render(ctx, 1.0)
        took = {}

        def behind():
            t = time.perf_counter()
            ctx.trace_rays(o, d)
            took["behind"] = time.perf_counter() - t

        th = threading.Thread(target=behind)
        th.start()
        time.sleep(0.05)
        t = time.perf_counter()
        got = other.trace_rays_noalloc(o, d)
        took["other"] = time.perf_counter() - t
        th.join(60)
        assert np.array_equal(got, want)
        assert took["behind"] > 0.5
        assert took["other"] < 0.5 * took["behind"], took

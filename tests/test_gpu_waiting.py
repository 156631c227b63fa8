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


def test_large_copies_of_others_while_one_waits(ctx, vtapi):
    """A readback behind a long render holds a ring; other contexts copy to and
    from the device meanwhile, and the readback itself comes back whole.  (Frames
    are set before: freeing one waits for the device.)"""
    import threading
    rng = np.random.default_rng(2)
    others = [vtapi.Context(0) for _ in range(2)]
    bad, got = [], {}

    def copies(c, k, w):
        for _ in range(3):
            a = rng.integers(0, 1 << 32, (1, w, 4), dtype=np.uint32).view(np.float32)
            c.write_accum(a)
            if not np.array_equal(c.read_accum().view(np.uint32), a.view(np.uint32)):
                bad.append((k, w))

    def behind():
        got["img"] = ctx.read_accum()

    for k, c in enumerate(others):
        c.set_frame((200000, 1 << 20)[k], 1)
        copies(c, k, (200000, 1 << 20)[k])
    long_render(ctx, 1.0)
    th = threading.Thread(target=behind)
    th.start()
    ts = [threading.Thread(target=copies, args=(c, k, (200000, 1 << 20)[k])) for k, c in enumerate(others)]
    for t in ts:
        t.start()
    for t in ts:
        t.join(60)
    th.join(60)
    for c in others:
        c.close()
    assert not bad
    assert np.array_equal(got["img"].view(np.uint32), ctx.read_accum().view(np.uint32))

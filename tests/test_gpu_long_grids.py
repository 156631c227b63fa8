"""Grids on both sides of the extent from which renders march step by step:
alone, in batches with small ones, under graph replays and into a cache."""
import time

import numpy as np
import pytest

from test_gpu_jump_march import bits_equal, workload_of

pytestmark = pytest.mark.gpu


def stats_image(c, wl):
    c.reset_accum()
    c.set_stats(True)
    c.render(wl.seed, 0, wl.spp)
    img = c.read_accum()
    c.set_stats(False)
    c.reset_accum()
    return img


@pytest.mark.parametrize("shape", [(12, 10, 900), (12, 901, 10), (901, 10, 12), (5, 6, 1016), (5, 6, 1017), (260, 20, 1300)])
def test_plain_equals_statistics(ctx, shape):
    from voxeltoy_amd import workloads
    wl = workload_of(shape, 0, 171, 111, np.random.default_rng(sum(shape)))
    workloads.load(ctx, wl)
    want = stats_image(ctx, wl)
    ctx.render(wl.seed, 0, wl.spp)
    assert bits_equal(ctx.read_accum(), want)


@pytest.mark.parametrize("other", [(12, 10, 900), (9, 6, 1000), (6, 5, 1500)])
def test_batch_with_a_long_grid(vtapi, other):
    from voxeltoy_amd import workloads
    rng = np.random.default_rng(other[2])
    wls = [workload_of(s, k % 3, 90 + k, 61, rng) for k, s in enumerate([(30, 40, 50), other, (16, 16, 16)])]
    ctxs = [vtapi.Context(0) for _ in wls]
    want = []
    for c, wl in zip(ctxs, wls):
        workloads.load(c, wl)
        want.append(stats_image(c, wl))
    b = vtapi.Batch(ctxs)
    try:
        for graph in (False, True, True, True):
            for c in ctxs:
                c.reset_accum()
            b.render([w.seed for w in wls], [w.spp for w in wls], graph=graph)
            for c, w in zip(ctxs, want):
                assert bits_equal(c.read_accum(), w)
        # the long grid goes, and the recorded graph with it
        small = workload_of((20, 21, 22), 0, 91, 61, rng)
        workloads.load(ctxs[1], small)
        want[1] = stats_image(ctxs[1], small)
        for c in ctxs:
            c.reset_accum()
        b.render([wls[0].seed, small.seed, wls[2].seed], [wls[0].spp, small.spp, wls[2].spp], graph=True)
        for c, w in zip(ctxs, want):
            assert bits_equal(c.read_accum(), w)
    finally:
        b.close()
        for c in ctxs:
            c.close()


@pytest.mark.parametrize("shape", [(40, 30, 900), (40, 30, 1000)])
def test_cache_render_with_the_cache_off(ctx, vtapi, shape):
    from voxeltoy_amd import workloads
    wl = workload_of(shape, 0, 171, 111, np.random.default_rng(shape[2]))
    wl.spp = 1
    workloads.load(ctx, wl)
    want = stats_image(ctx, wl)
    k = vtapi.RadianceCache(ctx, seed=1)
    k.render(wl.seed, 0, 1, cache_bounce=-1, train_paths=0)
    k.close()
    assert bits_equal(ctx.read_accum(), want)


@pytest.mark.parametrize("shape", [(20, 1500, 1500), (6, 7, 4096)])
def test_plain_is_no_slower_than_statistics(ctx, shape):
    from voxeltoy_amd import workloads
    wl = workload_of(shape, 0, 320, 200, np.random.default_rng(3))
    workloads.load(ctx, wl)

    def best():
        t = []
        for _ in range(8):
            a = time.perf_counter()
            ctx.render(wl.seed, 0, 2)
            ctx.synchronize()
            t.append(time.perf_counter() - a)
        return min(t[2:])

    plain = best()
    ctx.set_stats(True)
    counted = best()
    ctx.set_stats(False)
    assert plain < 1.2 * counted, (plain, counted)

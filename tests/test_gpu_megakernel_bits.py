"""The megakernel's block bits in LDS (the grid's own blocks, cut out of the
padded ones word by word): rows shorter and longer than a word, of whole words,
one block, slabs, and a grid whose bits do not fit in LDS.  Its image and its
counters are the wavefront's."""
import numpy as np
import pytest

from test_gpu_jump_march import bits_equal, workload_of

pytestmark = pytest.mark.gpu


# z, y, x extents; blocks of 4
@pytest.mark.parametrize("shape", [(1, 1, 1), (4, 4, 128), (3, 9, 131), (40, 12, 7), (33, 64, 257), (130, 126, 124),
                                   (9, 1030, 17), (1030, 5, 5), (320, 318, 322), (428, 425, 427), (432, 430, 436)])
def test_megakernel_equals_wavefront(ctx, shape):
    from voxeltoy_amd import workloads
    wl = workload_of(shape, 0, 161, 103, np.random.default_rng(sum(shape)))
    workloads.load(ctx, wl)
    try:
        ctx.render(wl.seed, 0, wl.spp)
        want = ctx.read_accum()
        ctx.set_render_mode(0)
        ctx.reset_accum()
        ctx.render(wl.seed, 0, wl.spp)
        assert bits_equal(ctx.read_accum(), want)
        counts = []
        for mode in (0, 1):
            ctx.set_render_mode(mode)
            ctx.set_stats(True)
            ctx.reset_accum()
            ctx.render(wl.seed, 0, wl.spp)
            assert bits_equal(ctx.read_accum(), want)
            st = ctx.stats()
            counts.append([st[k] for k in ("rays", "visits", "interactions", "samples")])
        assert counts[0] == counts[1]
    finally:
        ctx.set_stats(False)
        ctx.set_render_mode(1)


def test_megakernel_after_the_grid_changed(ctx):
    """New voxels of the same extents, and new extents, between two renders."""
    from voxeltoy_amd import workloads
    try:
        for k, shape in enumerate([(30, 20, 70), (30, 20, 70), (21, 33, 140), (30, 20, 70)]):
            wl = workload_of(shape, 0, 97, 65, np.random.default_rng(k))
            workloads.load(ctx, wl)
            images = []
            for mode in (1, 0):
                ctx.set_render_mode(mode)
                ctx.reset_accum()
                ctx.render(wl.seed, 0, wl.spp)
                images.append(ctx.read_accum())
            assert bits_equal(images[0], images[1])
    finally:
        ctx.set_render_mode(1)

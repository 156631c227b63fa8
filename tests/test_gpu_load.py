"""Grid upload: the one-pass conversion (bricks, block masks, codes) from offsets and from ids, into new and
kept buffers, and the checks of offsets and emissive lists on the device."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def grid(shape, rng, n_mat=5):
    ids = rng.integers(0, n_mat + 1, shape).astype(np.uint8) * (rng.random(shape) < 0.1)
    ids = ids.astype(np.uint8)
    ids.reshape(-1)[-1] = 1
    id_offset = np.full(256, -1, np.int32)
    id_offset[1:n_mat + 1] = rng.permutation(n_mat) * 8
    return ids, id_offset, rng.random(8 * n_mat).astype(np.float32)


def hits(ctx, shape, rng):
    n = 500
    o = rng.uniform(0.5, np.array(shape[::-1]) - 0.5, (n, 3)).astype(np.float32)
    d = rng.normal(size=(n, 3)).astype(np.float32)
    return ctx.trace_rays(o, d)


# one voxel; partial blocks, bricks and rows of cells on each axis; rows that are not a multiple of four
# voxels; two words of bits and more per wave; cells of 8 voxels
@pytest.mark.parametrize("shape", [(1, 1, 1), (4, 4, 4), (3, 5, 7), (8, 12, 16), (9, 13, 130), (65, 33, 62),
                                   (17, 64, 4), (270, 272, 275)])
def test_offsets_and_ids_convert_alike(ctx, shape):
    rng = np.random.default_rng(sum(shape))
    bmin, bmax = np.zeros(3), np.array(shape[::-1], np.float64)
    for _ in range(2):                                  # new buffers, then kept ones
        ids, id_offset, mat = grid(shape, rng)
        off = np.where(ids > 0, id_offset[ids], -1).astype(np.int32)
        em = np.flatnonzero(off >= 0)[:7].astype(np.int32)
        seed = int(rng.integers(1 << 30))
        ctx.set_volume(off, mat, emissive=em, bmin=bmin, bmax=bmax)
        assert np.array_equal(ctx.read_volume(), off)
        a = hits(ctx, shape, np.random.default_rng(seed))
        ctx.set_volume_u8(ids, id_offset, mat, emissive=em, bmin=bmin, bmax=bmax)
        assert np.array_equal(ctx.read_volume(), off)
        b = hits(ctx, shape, np.random.default_rng(seed))
        for x, y in zip(a, b) if isinstance(a, tuple) else [(a, b)]:
            assert np.array_equal(x, y)


def test_first_error_in_order(ctx, vtapi):
    off = np.full((5, 6, 7), -1, np.int32)
    off[1, 2, 3], off[4, 5, 6] = 24, 8
    mat = np.zeros(16, np.float32)

    def message(**kw):
        with pytest.raises(vtapi.VTError) as e:
            ctx.set_volume(off, mat, **kw)
        return str(e.value)

    ctx.set_volume(np.full((1, 2, 3), -1, np.int32), mat)
    off[0, 0, 1] = 16                                   # the first of the two bad offsets, before any emissive error
    assert "material offset 16 outside" in message(emissive=np.array([0], np.int32))
    off[0, 0, 1], off[1, 2, 3] = 0, 8
    assert "out of range at 1" in message(emissive=np.array([1, 210, 0], np.int32))
    assert "voxel 0 is empty" in message(emissive=np.array([1, 0, -1], np.int32))
    assert "out of range at 1" in message(emissive=np.array([1, -1, 0], np.int32))
    with pytest.raises(vtapi.VTError):
        ctx.read_volume()                               # a refused grid leaves no volume
    ctx.set_volume(off, mat, emissive=np.array([1, 209], np.int32))
    assert np.array_equal(ctx.read_volume(), off)

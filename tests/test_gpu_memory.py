"""Device memory that stays allocated after calls."""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def free_bytes():
    """By the runtime that the library loaded (torch brings another)."""
    with open("/proc/self/maps") as f:
        path = next(line.split()[-1] for line in f if "libamdhip64" in line)
    free, total = C.c_size_t(), C.c_size_t()
    assert C.CDLL(path).hipMemGetInfo(C.byref(free), C.byref(total)) == 0
    return free.value


def test_workspace_is_the_devices_not_each_contexts(vtapi):
    """Loading a 248^3 grid of offsets takes a workspace of 61 MB; the context
    itself keeps 21 MB (bricks, masks, codes)."""
    off = np.full((248, 248, 248), -1, np.int32)
    off[:4] = 0
    mat = np.array([0, 0, 0, 0, .5, .5, .5, 0], np.float32)
    ctxs = [vtapi.Context(0)]
    try:
        before = free_bytes()
        for _ in range(5):
            ctxs.append(vtapi.Context(0))
            ctxs[-1].set_volume(off, mat)
        used = before - free_bytes()
        assert used < 5 * 32e6 + 64e6, used
    finally:
        for c in ctxs:
            c.close()


def test_calls_that_share_the_workspace(vtapi, orc):
    """Threads with contexts of their own load, read back and pick at once."""
    import threading
    bad = []

    def work(k):
        try:
            rng = np.random.default_rng(k)
            mat = np.array([0, 0, 0, 0, .5, .5, .5, 0], np.float32)
            with vtapi.Context(0) as c:
                for i in range(4):
                    off = np.where(rng.random((40 + k, 61, 50 + i)) < 0.1, 0, -1).astype(np.int32)
                    c.set_volume(off, mat)
                    if not np.array_equal(c.read_volume(), off):
                        bad.append((k, i, "volume"))
                    lo, hi, _ = c.bounds()
                    o = rng.uniform(lo, hi, (20000, 3)).astype(np.float32)
                    d = rng.standard_normal((20000, 3)).astype(np.float32)
                    got = c.trace_rays(o, d)
                    if not np.array_equal(got[:2000], orc.OracleScene(off, mat).trace_rays(o[:2000], d[:2000])):
                        bad.append((k, i, "rays"))
        except BaseException as e:            # noqa: B902 - reported by the test
            bad.append(repr(e))

    ts = [threading.Thread(target=work, args=(k,)) for k in range(4)]
    for t in ts:
        t.start()
    for t in ts:
        t.join(60)
    assert not bad and not any(t.is_alive() for t in ts)


def test_vertices_without_triangles_take_no_memory(ctx, vtapi):
    """More vertices than the device could hold, none of them read."""
    off = np.full((8, 8, 8), -1, np.int32)
    off[0] = 0
    ctx.set_volume(off, np.array([0, 0, 0, 0, .5, .5, .5, 0], np.float32))
    occ = np.full((8, 8, 8), 7, np.uint8)
    rc = vtapi.lib().vt_voxelize(ctx._c, np.zeros(3, np.float32), 1 << 40, np.zeros(0, np.uint32), 0,
                                 np.eye(4, dtype=np.float32).reshape(-1), 0, 0, occ.ctypes.data)
    assert rc == 0, vtapi.lib().vt_last_error()
    assert not occ.any()
    assert np.array_equal(ctx.read_volume(), off)

"""Large copies between host arrays and the device (the staging ring of
vt_staging.h): sizes around its threshold, its chunks, its pieces and its ring
length, from one thread and from several, and after all contexts were gone."""
import threading

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# pixels of 16 bytes: 1 MiB threshold, 2 MiB chunks, 128 KiB pieces, 6 chunks in the ring
SIZES = [(65535, 1), (65536, 1), (65537, 1), (8192 * 9 + 1, 1), (131072, 1), (131071, 1), (131073, 1),
         (131072, 6), (131072, 7), (1920, 1080), (1021, 1777)]


def roundtrip(c, w, h, rng):
    c.set_frame(w, h)
    a = rng.integers(0, 1 << 32, (h, w, 4), dtype=np.uint32).view(np.float32)
    c.write_accum(a)
    got = c.read_accum()
    assert np.array_equal(got.view(np.uint32), a.view(np.uint32)), (w, h)


@pytest.mark.parametrize("w,h", SIZES)
def test_frame_roundtrip(ctx, w, h):
    roundtrip(ctx, w, h, np.random.default_rng(w))


def test_back_to_back_and_changing_sizes(ctx):
    rng = np.random.default_rng(5)
    for w, h in [(131072, 7), (65537, 1), (1920, 1080), (131073, 2), (640, 480)]:
        roundtrip(ctx, w, h, rng)


def test_several_threads_share_the_ring(vtapi):
    bad = []

    def work(k):
        try:
            rng = np.random.default_rng(k)
            with vtapi.Context(0) as c:
                for i in range(4):
                    roundtrip(c, *SIZES[(k + 3 * i) % len(SIZES)], rng)
        except BaseException as e:            # noqa: B902 - reported by the test
            bad.append(repr(e))

    ts = [threading.Thread(target=work, args=(k,)) for k in range(5)]
    for t in ts:
        t.start()
    for t in ts:
        t.join(60)
    assert not bad and not any(t.is_alive() for t in ts)


def test_ring_is_made_again_after_its_last_context(vtapi):
    for k in range(2):
        with vtapi.Context(0) as c:
            roundtrip(c, 1024, 512, np.random.default_rng(k))

"""The shorter exact quotients and roots of the kernels against IEEE arithmetic: every significand at both parities of
the exponent, random bit patterns, and the edges of the ranges in which they replace the operators."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def arguments():
    rng = np.random.default_rng(1)
    sig = np.arange(1 << 23, dtype=np.uint32)
    edges = np.array([0, 1, 0x007fffff, 0x00800000, 0x00800001, 0x7e7fffff, 0x7e800000, 0x7e800001, 0x7f7fffff,
                      0x7f800000, 0x7fc00000, (127 - 90) << 23, ((127 - 90) << 23) - 1, (127 - 100) << 23,
                      ((127 - 100) << 23) - 1], np.uint32)
    edges = np.concatenate([edges, edges | 0x80000000])
    return np.concatenate([sig | (127 << 23), sig | (128 << 23), rng.integers(0, 1 << 32, 1 << 21, dtype=np.uint32),
                           edges.astype(np.uint32)]).view(np.float32)


@pytest.mark.parametrize("fn", [0, 9, 10, 11, 12])
def test_exact(ctx, fn):
    a = arguments()
    if fn in (0, 10):
        a = np.abs(a)
    one, pi, two_pi = np.float32(1), np.float32(3.14159265359), np.float32(6.28318530718)
    with np.errstate(all="ignore"):
        want = {0: lambda: np.sqrt(a), 9: lambda: one / a, 10: lambda: one / np.sqrt(a), 11: lambda: a / pi,
                12: lambda: a / two_pi}[fn]()
    got = ctx.device_math(fn, a, a)
    assert ((got.view(np.uint32) == want.view(np.uint32)) | (np.isnan(got) & np.isnan(want))).all()

"""CPU emulation of the jump march (JumpState in voxeltoy_amd/csrc/vt_device.h)
against the oracle's raymarch (src/shaders/shared/dda.h:7-61): empty-cube codes
built as cell_codes_kernel builds them, positions from the real-line values
with the error bound, undecided jumps by the voxels they could skip and else
from the exact FP32 sums.  Every table
read must fall inside its table, the voxel a ray stops in must be the
oracle's, and every jump must move."""
import numpy as np
import pytest

F = np.float32
ULP24 = F(2.0 ** -24)
W1, W4 = F(2.5146484375e-4), F(1.005859375e-3)


def fma(a, b, c):
    """FP32 multiply-add with one rounding (the double product is exact; the
    double sum is exact for the magnitudes used here or rounds far below the
    march's error bound)."""
    return F(float(a) * float(b) + float(c))


def codes_of(occ, cg, top):
    """(padded cell codes, cube edges minus one per code)."""
    nz, ny, nx = occ.shape
    e = 1 << cg
    n = [-(-v // e) for v in (nx, ny, nz)]
    big = 1 << top
    up = [-(-v // big) * big for v in n]
    full = np.ones([v * e for v in up[::-1]], bool)
    full[:nz, :ny, :nx] = occ

    def any_in(k):
        return full.reshape(full.shape[0] // k, k, full.shape[1] // k, k, full.shape[2] // k, k).any((1, 3, 5))

    def spread(a, k):
        return a.repeat(k, 0).repeat(k, 1).repeat(k, 2)

    c1, c2, c3 = any_in(e), spread(any_in(2 * e), 2), spread(any_in(big * e), big)
    code = np.where(c1, 0, np.where(~c3, 3, np.where(~c2, 2, 1))).astype(np.uint8)
    out = np.zeros([v + 2 for v in n[::-1]], np.uint8)
    out[1:-1, 1:-1, 1:-1] = code[:n[2], :n[1], :n[0]]
    return out, [0, e - 1, 2 * e - 1, big * e - 1]


def padded_masks(occ):
    nz, ny, nx = occ.shape
    k = [(v + 3) // 4 for v in (nx, ny, nz)]
    full = np.ones([4 * (v + 2) for v in k[::-1]], bool)
    full[4:4 + nz, 4:4 + ny, 4:4 + nx] = occ
    return full.reshape(k[2] + 2, 4, k[1] + 2, 4, k[0] + 2, 4).transpose(0, 2, 4, 1, 3, 5).reshape(
        k[2] + 2, k[1] + 2, k[0] + 2, 64)


def sum_steps(X, a, ia, n):
    X, a = F(X), F(a)
    while n > 0:
        p = F(X + a)
        n -= 1
        if n == 0:
            return p
        X = F(p + a)
        n -= 1
        ub = int(X.view(np.uint32)) & 0x7F800000
        if n > 0 and ub == (int(p.view(np.uint32)) & 0x7F800000):
            end = np.uint32(ub + 0x00800000).view(F)
            r = min(int(F(F(end - X) * F(ia))) - 2, n)
            if r > 0:
                X = fma(F(r), F(F(X + a) - X), X)
                n -= r
    return X


def march(occ, tables, cg, res, bmin, bmax, o, d):
    """One ray: (stopped voxel or None when the start is outside, undecided jumps)."""
    code, edges, masks = tables
    ext = [F(1.0) / (F(bmax[i]) - F(bmin[i])) for i in range(3)]
    oo = [F(o[i]) + F(np.sign(F(d[i]))) * F(0.001) for i in range(3)]
    vo = [F(F(F(oo[i] - F(bmin[i])) * ext[i]) * F(res[i])) for i in range(3)]
    vp = [F(np.floor(v)) for v in vo]
    if any(v < 0 or v >= F(r) for v, r in zip(vp, res)):
        return None, 0
    dc = [F(1e-5) if F(1e-5) >= abs(F(v)) else F(v) for v in d]
    inc = [F(1.0) / v for v in dc]
    sg = [1 if v > 0 else -1 for v in dc]
    a = [F(abs(v)) for v in inc]
    X0 = [F(F(abs(F(F(F(vp[i] - vo[i]) + F(0.5)) + F(F(sg[i]) * F(0.5))))) * a[i]) for i in range(3)]
    if not all(F(2.0 ** -10) <= a[i] <= F(2e5) and X0[i] <= F(2e5) for i in range(3)):
        return "stepwise", 0
    ia = [F(1.0) / v for v in a]
    f = [-1 if s < 0 else 0 for s in sg]
    p = [int(vp[i]) ^ f[i] for i in range(3)]
    p0 = list(p)
    q = [fma(-X0[i], ia[i], F(p0[i] + 1)) for i in range(3)]
    c0 = F(ULP24 * F(2 * max(res) + 32))
    w1 = F(W1 * max(ia))
    undecided = 0
    for _ in range(sum(res) + 8):
        u = [p[i] ^ f[i] for i in range(3)]
        ci = [(u[i] + (1 << cg)) >> cg for i in range(3)]
        assert all(0 <= ci[i] < code.shape[2 - i] for i in range(3))
        c = code[ci[2], ci[1], ci[0]]
        edge = edges[c]
        if c == 0:
            bi = [(u[i] + 4) >> 2 for i in range(3)]
            assert all(0 <= bi[i] < masks.shape[2 - i] for i in range(3))
            m = masks[bi[2], bi[1], bi[0]]
            if not m.any():
                edge = 3
            elif m[(u[0] & 3) | ((u[1] & 3) << 2) | ((u[2] & 3) << 4)]:
                return tuple(u), undecided
        b = [v | edge for v in p]
        m = min(fma(F(b[i] - p0[i]), a[i], X0[i]) for i in range(3))
        w = fma(m, w1, W4)
        dl = fma(w, w, c0)
        pq = [F(fma(m, ia[i], q[i]) + dl) for i in range(3)]
        fr = [F(v - F(np.floor(v))) for v in pq]
        to = [int(np.floor(v)) for v in pq]
        if sorted(fr)[1] < dl + dl:
            d2 = dl + dl
            near = [fr[i] < d2 and to[i] > p[i] for i in range(3)]
            sums = all(near)
            if sum(near) == 2:
                am = max(a[i] for i in range(3) if near[i])
                e = [F(d2 * fma(am, ia[i], F(1))) for i in range(3)]
                sums = not max(e) < F(0.4) or any(
                    not near[i] and ((to[i] > p[i] and fr[i] < e[i]) or fr[i] > F(1) - e[i]) for i in range(3))
                for i in range(3):
                    if near[i] and not sums:
                        v = [(to[j] - (j == i)) ^ f[j] for j in range(3)]
                        bi = [(c + 4) >> 2 for c in v]
                        assert all(0 <= bi[j] < masks.shape[2 - j] for j in range(3))
                        sums = masks[bi[2], bi[1], bi[0]][(v[0] & 3) | ((v[1] & 3) << 2) | ((v[2] & 3) << 4)]
            if sums:
                undecided += 1
                t = [fma(F(b[i] - p0[i]), a[i], X0[i]) for i in range(3)]
                first = a[t.index(m)]
                cand = [i for i in range(3) if F(t[i] - m) <= F(d2 * F(a[i] + first))]
                m = min(sum_steps(X0[i], a[i], ia[i], b[i] - p0[i]) for i in cand)
                w = fma(m, w1, W4)
                dl = fma(w, w, c0)
                for i in range(3):
                    pv = F(fma(m, ia[i], q[i]) + dl)
                    to[i] = int(np.floor(pv))
                    if F(pv - F(np.floor(pv))) < dl + dl:
                        while to[i] > p[i] and sum_steps(X0[i], a[i], ia[i], to[i] - 1 - p0[i]) > m:
                            to[i] -= 1
        assert to != p and all(p[i] <= to[i] <= b[i] + 1 for i in range(3))
        p = to
    raise AssertionError("the march did not stop")


@pytest.mark.parametrize("shape,cg,top", [((16, 16, 16), 2, 2), ((20, 33, 65), 2, 2), ((7, 9, 230), 2, 3),
                                          ((48, 24, 64), 3, 2), ((40, 96, 33), 4, 2), ((1, 1, 5), 2, 2),
                                          ((2, 6, 4096), 2, 3)])
def test_jump_march_stops_where_the_oracle_does(orc, shape, cg, top):
    nz, ny, nx = shape
    res = (nx, ny, nz)
    rng = np.random.default_rng(nx + 1000 * cg)
    occ = rng.random(shape) < 0.002
    h = rng.integers(0, max(1, ny // 3) + 1, (nz, nx))
    occ |= np.arange(ny)[None, :, None] < h[:, None, :] * (rng.random((nz, 1, nx)) < 0.5)
    sc = orc.OracleScene(np.where(occ, 0, -1).astype(np.int32), np.zeros(7, np.float32))
    lo, hi = sc.bmin.astype(np.float64), sc.bmax.astype(np.float64)
    code, edges = codes_of(occ, cg, top)
    tables = (code, edges, padded_masks(occ))
    vs = (hi - lo) / res
    n = 260
    o = rng.uniform(lo, hi, (n, 3))
    d = rng.standard_normal((n, 3))
    d[:60] *= [1.0, 0.02, 1.0]                                     # grazing
    d[60:100, :] = np.eye(3)[rng.integers(0, 3, 40)] * rng.choice([-1.0, 1.0], (40, 1))
    d[100:140] = rng.choice([-1.0, 1.0], (40, 3)) * rng.integers(1, 4, (40, 3))   # ties of two and three axes
    o[80:140] = lo + rng.integers(0, np.array(res) + 1, (60, 3)) * vs             # from voxel corners
    o[200:, 1] = hi[1] - 1e-3 * vs[1]
    d[200:, 1] = -np.abs(d[200:, 1])
    # past voxel edges at distances from 1e-7 to 1e-3 voxels, half of them along steep axes
    near = (rng.integers(0, np.array(res) + 1, (60, 3)) + rng.normal(0, 1, (60, 3)) * 10.0 ** rng.uniform(-7, -3, (60, 1)))
    near[np.arange(60), rng.integers(0, 3, 60)] += 0.37
    d[140:200] = rng.standard_normal((60, 3))
    d[np.arange(140, 200), rng.integers(0, 3, 60)] *= 10.0 ** rng.uniform(-3.5, 0, 60)
    o[140:200] = lo + near * vs - d[140:200] / np.abs(d[140:200]).max(1, keepdims=True) * rng.uniform(0, 0.6, (60, 1)) * (hi - lo)
    d /= np.linalg.norm(d, axis=1, keepdims=True)
    d[::9] *= rng.choice([0.3, 4.0, 50.0], (len(d[::9]), 1))           # not unit
    o, d = o.astype(np.float32), d.astype(np.float32)
    want = sc.trace_rays(o, d)
    undecided = stepwise = 0
    for r in range(n):
        got, und = march(occ, tables, cg, res, sc.bmin, sc.bmax, o[r], d[r])
        undecided += und
        if got == "stepwise":
            stepwise += 1
        elif want[r, 4] < 0:
            assert got is None
        else:
            assert got == tuple(want[r, 1:4]), (r, o[r], d[r])
    assert stepwise < n // 8
    assert undecided > 0 or max(shape) < 8


def test_sum_steps_equals_the_adds_one_by_one():
    rng = np.random.default_rng(3)
    for t in range(400):
        d = F(max(1e-5, 2.0 ** -rng.uniform(0, 17))) if t % 3 else F((1 + rng.integers(0, 16)) / 64.0)
        a = F(1.0) / d
        if t % 4 == 0:                          # few mantissa bits: rounding ties
            a = (np.uint32(int(a.view(np.uint32)) & ~((1 << int(rng.integers(0, 20))) - 1))).view(F)
        X = F(rng.random() * float(a))
        n = int(rng.integers(0, 4200 if t % 2 else 300))
        ia = F(F(1.0) / a) * F(1 + (t % 5 - 2) * 2.0 ** -23)          # a reciprocal good to an ulp or two
        want = X
        for _ in range(n):
            want = F(want + a)
        assert sum_steps(X, a, ia, n) == want, (X, a, n)

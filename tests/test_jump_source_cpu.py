"""The jump march's own source (voxeltoy_amd/csrc/vt_jump.h: the codes' and the
masks' cubes, the real-line jumps and what settles the undecided ones), compiled
for the CPU with the address sanitizer, against the oracle's raymarch
(src/shaders/shared/dda.h:7-61)."""
import os
import struct
import subprocess

import numpy as np
import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
F = np.float32


@pytest.fixture(scope="module")
def exe(tmp_path_factory):
    out = str(tmp_path_factory.mktemp("jump") / "jump_march")
    b = subprocess.run(["g++", "-O2", "-g", "-std=c++17", "-ffp-contract=off", "-fsanitize=address", "-Wall",
                        "-Wno-unused-function", "-I", os.path.join(ROOT, "tests", "cpp", "host_hip"),
                        "-I", os.path.join(ROOT, "voxeltoy_amd", "csrc"),
                        os.path.join(ROOT, "tests", "cpp", "jump_march.cpp"), "-o", out], capture_output=True, text=True)
    assert b.returncode == 0, b.stderr
    return out


def queue_entries(o, d):
    """prepare_ray, queue_a and queue_b (vt_device.h): n x 6 floats."""
    o, d = o.astype(F), d.astype(F)
    dc = np.where(F(1e-5) >= np.abs(d), F(1e-5), d)
    return np.concatenate([o + np.sign(d) * F(0.001), F(1) / dc], 1).astype(F)


def march(exe, tmp_path, occ, bmin, bmax, rays):
    nz, ny, nx = occ.shape
    a, b = str(tmp_path / "in"), str(tmp_path / "out")
    with open(a, "wb") as f:
        f.write(struct.pack("4i", nx, ny, nz, len(rays)))
        f.write(np.asarray(bmin, F).tobytes() + np.asarray(bmax, F).tobytes())
        f.write(np.ascontiguousarray(occ, np.uint8).tobytes() + np.ascontiguousarray(rays, F).tobytes())
    r = subprocess.run([exe, a, b], capture_output=True, text=True, timeout=100)
    assert r.returncode == 0, r.stderr[-3000:]
    return np.fromfile(b, np.int32).reshape(-1, 4)


def rays_of(rng, lo, hi, res, n):
    """All directions; grazing; along an axis; ties from voxel corners; past
    voxel edges at 1e-7 to 1e-3 voxels, many along steep axes; down from the top;
    some not of unit length."""
    vs = (hi - lo) / res
    o = rng.uniform(lo, hi, (n, 3))
    d = rng.standard_normal((n, 3))
    k = np.arange(n) % 8
    d[k == 1] *= [1.0, 0.02, 1.0]
    m = k == 2
    d[m] = np.eye(3)[rng.integers(0, 3, m.sum())] * rng.choice([-1.0, 1.0], (m.sum(), 1))
    m = k == 3
    d[m] = rng.choice([-1.0, 1.0], (m.sum(), 3)) * rng.integers(1, 4, (m.sum(), 3))
    m = (k == 2) & (rng.random(n) < 0.5) | (k == 3)
    o[m] = lo + rng.integers(0, np.array(res) + 1, (m.sum(), 3)) * vs
    m = (k == 4) | (k == 5)
    w = m.sum()
    near = rng.integers(0, np.array(res) + 1, (w, 3)) + rng.normal(0, 1, (w, 3)) * 10.0 ** rng.uniform(-7, -3, (w, 1))
    near[np.arange(w), rng.integers(0, 3, w)] += 0.37
    dm = rng.standard_normal((w, 3))
    dm[np.arange(w), rng.integers(0, 3, w)] *= 10.0 ** rng.uniform(-3.5, 0, w)
    o[m] = lo + near * vs - dm / np.abs(dm).max(1, keepdims=True) * rng.uniform(0, 0.6, (w, 1)) * (hi - lo)
    d[m] = dm
    m = k == 6
    o[m, 1] = hi[1] - 1e-3 * vs[1]
    d[m, 1] = -np.abs(d[m, 1])
    d /= np.linalg.norm(d, axis=1, keepdims=True)
    d[::9] *= rng.choice([0.3, 4.0, 50.0], (len(d[::9]), 1))
    return o.astype(F), d.astype(F)


def compare(exe, tmp_path, orc, occ, o, d, least):
    sc = orc.OracleScene(np.where(occ, 0, -1).astype(np.int32), np.zeros(7, F))
    got = march(exe, tmp_path, occ, sc.bmin, sc.bmax, queue_entries(o, d))
    want = sc.trace_rays(o, d)
    outside = want[:, 4] < 0
    assert not (got[:, 0] < 0).any()
    assert (got[outside, 0] == 0).all() and (got[~outside, 0] != 0).all()
    ready = got[:, 0] == 1
    assert ready.sum() >= least
    wrong = np.flatnonzero(ready & (got[:, 1:] != want[:, 1:4]).any(1))
    assert len(wrong) == 0, (len(wrong), o[wrong[:3]], d[wrong[:3]], got[wrong[:3]], want[wrong[:3]])


# cells of 4 voxels with cubes of up to 4 and 8 cells, of 8 and of 16; extents around multiples of 4; slabs
@pytest.mark.parametrize("shape", [(16, 16, 16), (20, 33, 65), (7, 9, 230), (1, 1, 5), (2, 6, 4096), (270, 64, 275),
                                   (300, 300, 300), (97, 1, 130)])
@pytest.mark.parametrize("fill", [0.002, 0.03])
def test_march_stops_where_the_oracle_does(exe, tmp_path, orc, shape, fill):
    nz, ny, nx = shape
    rng = np.random.default_rng(nx + int(1000 * fill))
    occ = rng.random(shape) < fill
    h = rng.integers(0, max(1, ny // 3) + 1, (nz, nx))
    occ |= np.arange(ny)[None, :, None] < h[:, None, :] * (rng.random((nz, 1, nx)) < 0.5)
    lo = -500.0 * np.array([nx, ny, nz]) / max(shape)
    o, d = rays_of(rng, lo, -lo, (nx, ny, nz), 12000)
    compare(exe, tmp_path, orc, occ, o, d, 5000)


@pytest.mark.parametrize("edge,at", [(2, 0), (2, 1), (3, 0), (1, 0)])
def test_cubes_inside_blocks(exe, tmp_path, orc, edge, at):
    """Blocks with one voxel, row or corner filled, at every place: passages of
    2x2x2 voxels, aligned and not, inside occupied blocks."""
    rng = np.random.default_rng(edge + 10 * at)
    occ = np.zeros((48, 48, 48), bool)
    p = rng.integers(0, 12, (900, 3)) * 4 + rng.integers(0, 4 - edge + 1, (900, 3))
    for z, y, x in p:
        occ[z:z + edge, y:y + 1 + at, x:x + 1] = True
    o, d = rays_of(rng, np.full(3, -500.0), np.full(3, 500.0), (48, 48, 48), 24000)
    compare(exe, tmp_path, orc, occ, o, d, 10000)


@pytest.mark.parametrize("wall", [3970, 3971, 3972, 4092])
def test_far_end_of_the_longest_grid(exe, tmp_path, orc, wall):
    """4096 voxels an axis: the error bound passes one voxel near the 3970th
    step.  Rays along x whose y and z step together right before the step
    into a wall."""
    res = np.array([4096, 6, 6])
    occ = np.zeros(res[::-1], bool)
    occ[:, :, wall] = True
    rng = np.random.default_rng(wall)
    n = 4000
    hi = 500.0 * res / 4096
    vs = 1000.0 / 4096
    p = np.concatenate([rng.uniform(0, 1, (n, 1)), rng.uniform(2, 3, (n, 2))], 1)
    p[::2, 2] = p[::2, 1]
    rest = wall - p[:, 0] - 10.0 ** rng.uniform(-5, -2, n)
    slope = (np.ceil(p[:, 1:]) - p[:, 1:]) / rest[:, None]
    d = np.concatenate([np.ones((n, 1)), slope], 1)
    d *= rng.uniform(0.7, 1.4, (n, 1))                  # steps that are no round numbers
    o = p * vs - hi - np.sign(d) * 0.001
    compare(exe, tmp_path, orc, occ, o.astype(F), d.astype(F), n // 2)

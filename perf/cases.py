"""What the library is timed on: renders, voxelizations, picks and radiance-cache
calls through the public ctypes binding (voxeltoy_amd.api), from a single
picking ray to a 16-pass megapixel still.

A case is a dict with a "kind" (which call a user's program makes) and its
sizes.  Scenes are made from the seed as the repository's workloads make them:
value-noise terrain with boxes, 70/20/10 Lambert/metal/emissive materials, a
sky-and-sun image or a gradient environment, orbiting cameras.
"""
import math

import numpy as np
import torch

from voxeltoy_amd import api, scenes, workloads

SKY_TOP, SKY_BOTTOM = (1.6, 1.7, 1.9), (0.35, 0.3, 0.25)


def listed():
    return [
        # picking on a mouse move: one ray against a small loaded model, records back on the host
        {"name": "pick_one_ray", "kind": "pick", "nx": 126, "ny": 20, "nz": 126, "rays": 1},
        # the small preview: four passes of a thumbnail-sized frame over a 64^3 model
        {"name": "preview_256", "kind": "render", "nx": 64, "ny": 64, "nz": 64, "width": 256, "height": 256,
         "spp": 4, "bounces": 4, "lens": 0, "env": "white", "fp64": False},
        # an odd window over an odd grid, orthographic, with the double-precision sums kept for a reference image
        {"name": "ragged_fp64", "kind": "render", "nx": 201, "ny": 93, "nz": 157, "width": 643, "height": 357,
         "spp": 3, "bounces": 5, "lens": 2, "env": "gradient", "fp64": True},
        # one frame of the interactive viewer: one more pass of a full-HD progressive render, then the image
        {"name": "frame_1080p", "kind": "frame", "n": 256, "width": 1920, "height": 1080, "bounces": 8},
        # the full-shading still: 256^3, thin lens, image environment, 16 passes of 8 bounces
        {"name": "still_1024_16spp", "kind": "still", "n": 256, "width": 1024, "height": 1024, "spp": 16,
         "bounces": 8},
        # opening a scene: the int32 material-offset grid uploaded, then its first small frame
        {"name": "open_scene_256", "kind": "open", "nx": 256, "ny": 256, "nz": 256, "width": 960, "height": 540,
         "spp": 1, "bounces": 4},
        # a mesh imported into a large grid and rendered
        {"name": "mesh_512_1080p", "kind": "mesh", "triangles": 200000, "res": 512, "mode": 0, "width": 1920,
         "height": 1080, "spp": 8, "bounces": 6},
        # conservative voxelization alone, with the dense occupancy returned
        {"name": "voxelize_fat_256", "kind": "voxelize", "triangles": 50001, "res": 256, "mode": 1},
        # a batch of unlike scenes through one recorded graph
        {"name": "batch_16", "kind": "batch", "scenes": 16, "n_lo": 32, "n_hi": 200, "res_lo": 128, "res_hi": 700,
         "spp_hi": 24, "bounces": 4},
        # one viewer frame that ends paths into the radiance cache and trains it
        {"name": "cached_frame_1080p", "kind": "cached", "n": 256, "width": 1920, "height": 1080, "bounces": 8,
         "cache_bounce": 2, "train_paths": 65536, "train_extra": 1},
        # a gradient of the cache's network over one frame's training samples
        {"name": "cache_gradient_50k", "kind": "gradient", "samples": 50001},
        # the queries of one frame answered by the network
        {"name": "cache_infer_400k", "kind": "infer", "samples": 411517},
    ]


def draw(rng):
    def log(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    kind = rng.choice(["pick", "render", "render", "frame", "still", "open", "mesh", "voxelize", "batch", "cached",
                       "gradient", "infer"])
    if kind == "pick":
        return {"kind": kind, "nx": log(20, 400), "ny": log(16, 300), "nz": log(20, 400), "rays": log(1, 16384)}
    if kind == "render":
        return {"kind": kind, "nx": log(17, 320), "ny": log(17, 320), "nz": log(17, 320), "width": log(40, 1600),
                "height": log(40, 1000), "spp": log(1, 6), "bounces": rng.randint(1, 8), "lens": rng.randint(0, 2),
                "env": rng.choice(["white", "gradient", "image"]), "fp64": rng.random() < 0.3}
    if kind == "frame":
        return {"kind": kind, "n": log(64, 320), "width": log(320, 1920), "height": log(200, 1080),
                "bounces": rng.randint(2, 8)}
    if kind == "still":
        return {"kind": kind, "n": log(64, 256), "width": log(200, 1024), "height": log(200, 1024),
                "spp": rng.randint(4, 16), "bounces": rng.randint(2, 8)}
    if kind == "open":
        return {"kind": kind, "nx": log(33, 256), "ny": log(33, 256), "nz": log(33, 256), "width": log(64, 960),
                "height": log(64, 540), "spp": 1, "bounces": rng.randint(1, 4)}
    if kind == "mesh":
        return {"kind": kind, "triangles": log(1000, 200000), "res": log(64, 512), "mode": rng.randint(0, 1),
                "width": log(320, 1920), "height": log(200, 1080), "spp": rng.randint(1, 8),
                "bounces": rng.randint(1, 6)}
    if kind == "voxelize":
        return {"kind": kind, "triangles": log(12, 200000), "res": log(32, 320), "mode": rng.randint(0, 1)}
    if kind == "batch":
        return {"kind": kind, "scenes": rng.randint(2, 16), "n_lo": 32, "n_hi": log(64, 200), "res_lo": 64,
                "res_hi": log(128, 700), "spp_hi": rng.randint(1, 24), "bounces": rng.randint(1, 6)}
    if kind == "cached":
        return {"kind": kind, "n": log(64, 256), "width": log(320, 1920), "height": log(200, 1080),
                "bounces": rng.randint(4, 8), "cache_bounce": rng.randint(1, 3), "train_paths": log(4096, 65536),
                "train_extra": 1}
    return {"kind": kind, "samples": log(16, 262144)}


# ---- inputs -----------------------------------------------------------------------------------

def _scene(rng, nx, ny, nz, n_ids=40, n_boxes=24):
    """Value-noise terrain and boxes on any grid, materials 70/20/10."""
    m = max(nx, nz)
    h = 0.6 * scenes.value_noise_2d(rng, m, max(2, m // 40)) + 0.4 * scenes.value_noise_2d(rng, m, max(3, m // 15))
    h = (h[:nz, :nx] * 0.35 + 0.05) * ny
    occ = np.arange(ny)[None, :, None] < h[:, None, :]
    size = np.array([nx, ny, nz])
    for _ in range(n_boxes):
        s = rng.integers(np.maximum(1, size // 32), np.maximum(2, size // 8))
        p = rng.integers(0, size - s)
        occ[p[2]:p[2] + s[2], p[1]:p[1] + s[1], p[0]:p[0] + s[0]] = True
    n_lam, n_met = int(round(0.7 * n_ids)), int(round(0.2 * n_ids))
    recs = [scenes.lambert((0, 0, 0), rng.uniform(0.2, 0.8, 3)) for _ in range(n_lam)]
    recs += [scenes.metal((0, 0, 0), rng.uniform(0.5, 0.95, 3), rng.uniform(0.05, 0.6)) for _ in range(n_met)]
    recs += [scenes.lambert(rng.lognormal(1.0, 0.5) * rng.uniform(0.7, 1.0, 3), rng.uniform(0.2, 0.8, 3))
             for _ in range(n_ids - n_lam - n_met)]
    mat, offs = scenes.build_materials(recs)
    id_offset = np.full(256, -1, np.int32)
    id_offset[1:n_ids + 1] = offs
    ids = np.where(occ, rng.integers(1, n_ids + 1, size=occ.shape, dtype=np.uint8), 0).astype(np.uint8)
    sc = scenes.Scene(ids, id_offset, mat)
    sc.emissive = api.prune_emissive(sc.offsets(), scenes.emissive_list(ids, id_offset, mat))
    return sc


def _camera(rng, shape, width, height, lens):
    bmin, bmax = workloads.reference_bounds(shape)
    extent = float(np.max(bmax - bmin))
    cam = scenes.orbit_camera(bmin, bmax, math.radians(rng.uniform(105, 140)), rng.uniform(0, 2 * math.pi), width,
                              height, lens_model=lens, lens_radius=0.02 * extent)
    if lens == 1:
        cam.focal_distance = float(np.linalg.norm(cam.target - cam.eye)) * rng.uniform(0.8, 1.1)
    return cam, bmin, bmax


def _workload(rng, sc, width, height, spp, bounces, lens, env, seed):
    cam, bmin, bmax = _camera(rng, sc.shape, width, height, lens)
    wl = workloads.Workload("case", sc, cam, width, height, spp=spp, bounces=bounces, seed=seed, bmin=bmin, bmax=bmax)
    if env != "white":
        wl.env_top, wl.env_bottom = SKY_TOP, SKY_BOTTOM
    if env == "image":
        wl.env_image = scenes.sky_environment(seed + 3, 512, 256)
        wl.cdf = api.env_build_cdf(wl.env_image)
        wl.env_rotation = float(rng.uniform(0, 2 * math.pi))
    return wl


def _batch_sizes(case):
    """Grid edge, image edge and passes of each scene, log-uniform; they belong to the case, not to the seed."""
    rng = np.random.default_rng([case["scenes"], case["n_hi"], case["res_hi"], case["spp_hi"]])
    lo = np.log([case["n_lo"], case["res_lo"], 1])
    hi = np.log([case["n_hi"], case["res_hi"], case["spp_hi"]])
    return np.rint(np.exp(rng.uniform(lo, hi, (case["scenes"], 3)))).astype(int).tolist()


def _mesh(rng, triangles):
    """A closed displaced sphere of about `triangles` triangles, shared vertices."""
    nv = max(2, int(round(math.sqrt(triangles / 4.0))))
    nu = max(3, int(round(triangles / (2.0 * nv))))
    u = np.arange(nu) * (2 * math.pi / nu)
    v = (np.arange(nv + 1) / nv) * math.pi
    d = np.stack([np.sin(v)[:, None] * np.cos(u), np.cos(v)[:, None] * np.ones(nu), np.sin(v)[:, None] * np.sin(u)],
                 -1).reshape(-1, 3)
    k, ph = rng.standard_normal((8, 3)), rng.uniform(0, 2 * math.pi, 8)
    noise = sum(np.sin(d @ (k[i] * (1.5 + i)) + ph[i]) / (1 + i) for i in range(8))
    verts = (d * (1 + 0.05 * noise / np.abs(noise).max())[:, None]).astype(np.float32)
    a = (np.arange(nv)[:, None] * nu + np.arange(nu)[None, :]).reshape(-1)
    b = (np.arange(nv)[:, None] * nu + (np.arange(nu)[None, :] + 1) % nu).reshape(-1)
    tris = np.concatenate([np.stack([a, b, a + nu], 1), np.stack([b, b + nu, a + nu], 1)]).astype(np.uint32)
    return verts, np.ascontiguousarray(tris)


def _queries(rng, n):
    """Cache queries: positions in the unit cube, unit directions and axis normals mapped to [0, 1], albedo."""
    d = rng.standard_normal((n, 3))
    d /= np.linalg.norm(d, axis=1, keepdims=True)
    nrm = np.zeros((n, 3))
    nrm[np.arange(n), rng.integers(0, 3, n)] = rng.choice([-1.0, 1.0], n)
    raw = np.concatenate([rng.random((n, 3)), (d + 1) / 2, (nrm + 1) / 2, rng.uniform(0.2, 0.8, (n, 3))], 1)
    return raw.astype(np.float32)


def _network(rng):
    """Weights of a network in use: He-uniform layers with small biases."""
    p = []
    for out, inp in [(64, 288)] + [(64, 64)] * 4 + [(3, 64)]:
        p += [rng.uniform(-1, 1, out * inp) * math.sqrt(6.0 / inp), rng.uniform(-0.05, 0.05, out)]
    return np.concatenate(p).astype(np.float32)


def _cache_inputs(case, seed):
    rng = np.random.default_rng(seed)
    raw = _queries(rng, case["samples"])
    return _network(rng), raw, rng.lognormal(0.0, 1.0, (case["samples"], 3)).astype(np.float32)


# ---- a user's program ---------------------------------------------------------------------------

def prepare(case, seed):
    rng = np.random.default_rng(seed)
    kind = case["kind"]
    s = {"case": case, "seed": seed % 100003 + 1, "n": 0}
    if kind == "batch":
        ctxs, counts = [], []
        for i, (n, res, spp) in enumerate(_batch_sizes(case)):
            wl = _workload(rng, scenes.mixed_scene(rng, n, float(rng.uniform(0.05, 0.6))), res, res, spp,
                           case["bounces"], 0, "gradient", s["seed"] + i)
            wl.scene.emissive = api.prune_emissive(wl.scene.offsets(), wl.scene.emissive)
            ctxs.append(api.Context(0))
            workloads.load(ctxs[-1], wl)
            counts.append(spp)
        s.update(ctxs=ctxs, counts=counts, batch=api.Batch(ctxs), seeds=[s["seed"] + i for i in range(len(ctxs))])
        return s
    ctx = s["ctx"] = api.Context(0)
    if kind in ("gradient", "infer"):
        params, s["raw"], s["target"] = _cache_inputs(case, seed)
        s["cache"] = api.RadianceCache(ctx, seed=1)
        s["cache"].set_params(params)
        return s
    if kind in ("mesh", "voxelize"):
        res = case["res"]
        s["verts"], s["tris"] = _mesh(rng, case["triangles"])
        s["M"] = api.mesh_transform(s["verts"].min(0), s["verts"].max(0), [res] * 3)
        mat = np.asarray(scenes.lambert((0, 0, 0), (0.7, 0.65, 0.6)), np.float32)
        empty = scenes.Scene(np.zeros((res,) * 3, np.uint8), np.full(256, -1, np.int32), mat)
        if kind == "voxelize":
            ctx.set_volume_u8(empty.ids, empty.id_offset, mat)
            return s
        wl = _workload(rng, empty, case["width"], case["height"], case["spp"], case["bounces"], 0, "gradient",
                       s["seed"])
    elif kind in ("frame", "still", "cached"):
        wl = workloads.full(case["width"], case["height"], seed_scene=int(rng.integers(1, 1 << 30)), n=case["n"],
                            env_w=512, env_h=256, bounces=case["bounces"])
    elif kind == "pick":
        sc = _scene(rng, case["nx"], case["ny"], case["nz"])
        ctx.set_volume_u8(sc.ids, sc.id_offset, sc.mat, sc.emissive)
        lo, hi = workloads.reference_bounds(sc.shape)
        # rays as picking makes them: from where the view ray enters the bounds, towards a point of the volume
        o = rng.uniform(0.02, 0.98, (case["rays"], 3)) * (hi - lo) + lo
        o[:, 1] = hi[1] - 0.01 * (hi[1] - lo[1])
        d = rng.uniform(0.0, 1.0, o.shape) * (hi - lo) * np.array([1.0, 0.5, 1.0]) + lo - o
        s["o"], s["d"] = o.astype(np.float32), (d / np.linalg.norm(d, axis=1, keepdims=True)).astype(np.float32)
        return s
    else:
        sc = _scene(rng, case["nx"], case["ny"], case["nz"])
        wl = _workload(rng, sc, case["width"], case["height"], case["spp"], case["bounces"], case.get("lens", 0),
                       case.get("env", "gradient"), s["seed"])
        if kind == "open":
            s["offsets"], s["mat"], s["emissive"] = sc.offsets(), sc.mat, sc.emissive
    workloads.load(ctx, wl, fp64=bool(case.get("fp64")))
    if kind == "cached":
        s["cache"] = api.RadianceCache(ctx, seed=s["seed"])
    return s


def run(s):
    case, ctx, kind = s["case"], s.get("ctx"), s["case"]["kind"]
    if kind == "pick":
        return ctx.trace_rays_noalloc(s["o"], s["d"])
    if kind == "infer":
        return s["cache"].infer(s["raw"])
    if kind == "gradient":
        g, loss = s["cache"].gradient(s["raw"], s["target"])
        return {"grad": g, "loss": loss}
    if kind == "voxelize":
        return ctx.voxelize(s["verts"], s["tris"], s["M"], mode=case["mode"], material_offset=0)
    if kind == "batch":
        for c in s["ctxs"]:
            c.reset_accum()
        s["batch"].render(s["seeds"], s["counts"], graph=True)
        return [c.read_accum() for c in s["ctxs"]]
    if kind == "frame":       # the viewer goes on: one pass more each time
        ctx.render(s["seed"], s["n"], 1)
        s["n"] += 1
        return ctx.read_accum()
    if kind == "cached":      # one Adam step over the frame's samples
        s["cache"].render(s["seed"], s["n"], 1, cache_bounce=case["cache_bounce"], train_paths=case["train_paths"],
                          train_extra=case["train_extra"], batch=1 << 18)
        s["n"] += 1
        return {"image": ctx.read_accum(), "params": s["cache"].params()}
    if kind == "open":
        ctx.set_volume(s["offsets"], s["mat"], s["emissive"])
    if kind == "mesh":
        ctx.voxelize(s["verts"], s["tris"], s["M"], mode=case["mode"], material_offset=0, want_occupancy=False)
    ctx.reset_accum()
    ctx.render(s["seed"], 0, case["spp"])
    if case.get("fp64"):
        return {"mean": ctx.read_accum(), "sum": ctx.read_sum64()}
    return ctx.read_accum()


# ---- what a pass cannot do without ----------------------------------------------------------------

def work(case):
    """Renders: the grid's bits and the frame once, and per traced ray (a
    sample's camera ray and, on average, about two vertices with a shadow and
    a continuation ray each) the voxel steps of a quarter of the grid's edge
    at ten operations, and about 300 operations of shading."""
    kind = case["kind"]
    if kind in ("gradient", "infer"):
        n = case["samples"]
        return {"bytes": n * 60.0, "flops": n * 70016.0 * (3 if kind == "gradient" else 1)}
    if kind == "pick":
        edge = max(case["nx"], case["ny"], case["nz"])
        return {"bytes": case["rays"] * 56.0, "flops": case["rays"] * (edge * 0.5 * 10 + 100)}
    if kind == "voxelize":
        return {"bytes": case["triangles"] * 48.0 + case["res"] ** 3, "flops": case["triangles"] * 400.0}
    if kind == "batch":
        sizes = _batch_sizes(case)
        edge = math.sqrt(case["n_lo"] * case["n_hi"])
        pixels, samples = (sum(r * r * (k if each else 1) for _, r, k in sizes) for each in (False, True))
        grid = sum(n ** 3 for n, _, _ in sizes) / 8.0
    else:
        pixels = case["width"] * case["height"]
        samples = pixels * case.get("spp", 1)
        dims = [case.get(k, case.get("n", case.get("res"))) for k in ("nx", "ny", "nz")]
        edge, grid = max(dims), dims[0] * dims[1] * dims[2] / 8.0
    extra = 0.0
    if kind == "open":
        extra = grid * 8 * 4
    if kind == "mesh":
        extra = case["triangles"] * 48.0
    rays = samples * (1 + 2 * min(2.2, case["bounces"]))
    return {"bytes": pixels * (40.0 if case.get("fp64") else 16.0) + grid + extra,
            "flops": rays * (edge * 0.25 * 10 + 300)}


# ---- results in 64 bits ------------------------------------------------------------------------------

def exact(case, seed):
    """The network's outputs and gradient in 64 bits.  An image has no such
    value: its random choices and voxel marches are defined in 32 bits."""
    if case["kind"] not in ("infer", "gradient"):
        return None
    params, raw, target = (torch.from_numpy(a).cuda().double() for a in _cache_inputs(case, seed))
    layers, at = [], 0
    for out, inp in [(64, 288)] + [(64, 64)] * 4 + [(3, 64)]:
        w = params[at:at + out * inp].view(out, inp).clone().requires_grad_()
        b = params[at + out * inp:at + out * inp + out].clone().requires_grad_()
        layers.append((w, b))
        at += out * (inp + 1)
    ys, loss, n = [], 0.0, len(raw)
    for lo in range(0, n, 65536):
        a = math.pi * raw[lo:lo + 65536, :, None] * 2.0 ** torch.arange(12, device="cuda", dtype=torch.float64)
        x = torch.stack([torch.sin(a), torch.cos(a)], -1).reshape(len(a), 288)
        for k, (w, b) in enumerate(layers):
            x = x @ w.t() + b
            x = torch.relu(x) if k < 5 else x
        ys.append(x.detach())
        if case["kind"] == "gradient":
            part = ((x - target[lo:lo + 65536]) ** 2 / (x.detach() ** 2 + 0.01)).sum() / (3 * n)
            part.backward()
            loss += float(part.detach())
    if case["kind"] == "infer":
        return torch.cat(ys)
    return {"grad": torch.cat([t.grad.reshape(-1) for wb in layers for t in wb]), "loss": loss}

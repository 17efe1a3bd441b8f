"""What a user of the renderer has it do, as cases that can be timed: batched ray queries, renders
(previews, full frames, odd sizes, direct lighting, every material under a sky, guided), batches of
images, the learned proposal alone, and a device BVH build with queries on the new tree.

Sizes are those of the workloads in spica_amd/configs.py, of the tests and of bench.py, or lie
between them.  Everything goes through the public handles of spica_amd.render.
"""
import math

import numpy as np
import torch

from spica_amd import _abi, configs, render

# The network of the learned proposal: 7 inputs in 32 bins each, four hidden layers, 8 lobes of 5.
LAYERS = [(64, 224), (64, 64), (64, 64), (64, 64), (40, 64)]


def listed():
    return [
        # picking and probe rays of an editor: few rays, a small scene, one answer at once
        {"name": "trace_pick", "kind": "trace", "scene": "cornell", "spheres": 0, "rays": 257, "any_hit": False},
        # closest hits for a caller that shades by itself: camera, uniform and scattered rays on the sphere field
        {"name": "trace_field", "kind": "trace", "scene": "field", "spheres": 512, "rays": 2_000_003, "any_hit": False},
        # visibility between two points (baking, ambient occlusion): bounded any-hit rays
        {"name": "occlude_field", "kind": "trace", "scene": "field", "spheres": 128, "rays": 300_007, "any_hit": True},
        # the smallest render: a preview tile while a scene is edited
        {"name": "render_preview", "kind": "render", "scene": "cornell", "spheres": 0, "width": 64, "height": 64,
         "spp": 4, "queue": 0, "integrator": "path"},
        # the Cornell box at its configured size, default options
        {"name": "render_cornell", "kind": "render", "scene": "cornell", "spheres": 0, "width": 256, "height": 256,
         "spp": 64, "queue": 0, "integrator": "path"},
        # the full sphere-field frame, many paths in flight
        {"name": "render_field", "kind": "render", "scene": "field", "spheres": 512, "width": 1920, "height": 1080,
         "spp": 32, "queue": 1 << 26, "integrator": "path"},
        # every BSDF kind under a sky, an odd film, default options
        {"name": "render_wide", "kind": "render", "scene": "wide", "spheres": 200, "width": 301, "height": 223,
         "spp": 12, "queue": 0, "integrator": "path"},
        # the occluded glossy scene with the proposal trained on the render's own first samples
        {"name": "render_guided", "kind": "render", "scene": "glossy", "spheres": 512, "width": 640, "height": 360,
         "spp": 96, "queue": 1 << 22, "integrator": "path", "train_spp": 32},
        # a batch of uneven images, each its own scene, film and sample count
        {"name": "batch_fields", "kind": "batch", "images": 8, "spheres": 512, "res": 512, "spp": 64, "queue": 1 << 22},
        # the proposal's loss gradient on a full training batch
        {"name": "guide_grad", "kind": "guide_grad", "samples": 1 << 18},
        # directions and densities of the proposal at given vertices
        {"name": "guide_sample", "kind": "guide_sample", "samples": 100_003},
        # a changed scene: the BVH built on the device, then a query on the new tree
        {"name": "build_trace", "kind": "build", "scene": "field", "spheres": 256, "rays": 65_536},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["trace", "trace", "render", "render", "render", "guided", "batch", "guide_grad", "guide_sample",
                       "build"])
    if kind == "trace":
        scene = rng.choice(["cornell", "field", "field", "glossy"])
        return {"kind": "trace", "scene": scene, "spheres": 0 if scene == "cornell" else _log_int(rng, 8, 512),
                "rays": _log_int(rng, 1, 2_000_000), "any_hit": rng.random() < 0.4}
    if kind == "render":
        scene = rng.choice(["cornell", "field", "field", "wide", "glossy"])
        w, h = _log_int(rng, 33, 1280), _log_int(rng, 31, 720)
        spp = max(1, min(_log_int(rng, 1, 64), 20_000_000 // (w * h)))
        return {"kind": "render", "scene": scene, "spheres": 0 if scene == "cornell" else _log_int(rng, 16, 512),
                "width": w, "height": h, "spp": spp, "queue": rng.choice([0, 0, 1 << 16, 1 << 20, 1 << 23]),
                "integrator": rng.choice(["path", "path", "direct"])}
    if kind == "guided":
        w, h = _log_int(rng, 65, 640), _log_int(rng, 63, 360)
        return {"kind": "render", "scene": "glossy", "spheres": _log_int(rng, 32, 512), "width": w, "height": h,
                "spp": rng.randint(17, 64), "queue": rng.choice([0, 1 << 20]), "integrator": "path",
                "train_spp": 8 * rng.randint(1, 4)}
    if kind == "batch":
        return {"kind": "batch", "images": rng.randint(2, 8), "spheres": _log_int(rng, 32, 512),
                "res": _log_int(rng, 64, 512), "spp": rng.randint(16, 64), "queue": rng.choice([0, 1 << 20, 1 << 22])}
    if kind == "build":
        return {"kind": "build", "scene": rng.choice(["field", "glossy"]), "spheres": _log_int(rng, 2, 256),
                "rays": _log_int(rng, 1, 65_536)}
    return {"kind": kind, "samples": _log_int(rng, 64, 1 << 18 if kind == "guide_grad" else 100_003)}


# ---- scenes and inputs ---------------------------------------------------------------------------
def _workload(case, seed):
    """The scene, camera and integrator settings of a trace, render or build case; for a case with
    spheres the seed draws them."""
    w, h, spp = case.get("width", 640), case.get("height", 360), case.get("spp", 1)
    if case["scene"] == "cornell":
        wl = configs.cornell_box(w, h, spp)
        wl.seed = seed
        return wl
    if case["scene"] == "glossy":
        return configs.c3_occluded_glossy(w, h, spp, seed=seed, n_spheres=case["spheres"])
    if case["scene"] == "wide":
        scene, _ = configs.sphere_field(seed, case["spheres"], mix=configs.WIDE_MIX)
        scene.set_envmap(configs.sky_envmap(256, 128, sun=50.0),
                         to_world=np.array([[1, 0, 0, 0], [0, 0, 1, 0], [0, 1, 0, 0], [0, 0, 0, 1]], float), radius=60.0)
        cam = configs.c1_spheres(w, h, n_spheres=0).camera
        return configs.Workload("every BSDF under a sky", scene, cam, spp, 16, _abi.SPK_SAMPLER_SOBOL, seed)
    return configs.c1_spheres(w, h, spp, seed=seed, n_spheres=case["spheres"])


def _unit(v):
    return v / v.norm(dim=1, keepdim=True)


def _rays(wl, n, seed, device):
    """A third camera rays in pixel order, a third uniform origins and directions in the scene box,
    a third leaving random points of the scene's triangles (the rays of a scattering vertex)."""
    g = torch.Generator(device=device).manual_seed(int(seed))
    rand = lambda *s: torch.rand(*s, generator=g, device=device, dtype=torch.float64)  # noqa: E731
    verts = torch.from_numpy(wl.scene.freeze()["verts"]).to(device).double()
    lo, hi = verts.amin(dim=(0, 1)), verts.amax(dim=(0, 1))
    n1, n2 = (n + 2) // 3, n // 3
    n3 = n - n1 - n2
    cam = wl.camera
    m = torch.from_numpy(cam.to_world).to(device)
    t = math.tan(math.radians(cam.fov_deg) / 2.0)
    pix = torch.arange(n1, device=device, dtype=torch.float64) * (cam.width * cam.height / max(n1, 1))
    px, py = torch.remainder(pix, cam.width), torch.floor(pix / cam.width) + rand(n1)
    dc = torch.stack([(2 * px / cam.width - 1) * cam.width / cam.height * t, (1 - 2 * py / cam.height) * t,
                      torch.ones_like(px)], 1)
    d1, o1 = _unit(dc @ m[:3, :3].T), m[:3, 3].expand(n1, 3)
    o2 = lo + (hi - lo) * rand(n2, 3)
    d2 = _unit(torch.randn(n2, 3, generator=g, device=device, dtype=torch.float64))
    tri = verts[(rand(n3) * len(verts)).long().clamp(max=len(verts) - 1)]
    b = torch.sqrt(rand(n3, 1))
    c = rand(n3, 1)
    nrm = _unit(torch.linalg.cross(tri[:, 1] - tri[:, 0], tri[:, 2] - tri[:, 0]))
    o3 = (1 - b) * tri[:, 0] + b * (1 - c) * tri[:, 1] + b * c * tri[:, 2] + 1e-3 * nrm
    d3 = _unit(nrm + 0.999 * _unit(torch.randn(n3, 3, generator=g, device=device, dtype=torch.float64)))
    org = torch.cat([o1, o2, o3]).float().contiguous()
    dirv = torch.cat([d1, d2, d3]).float().contiguous()
    # visibility queries between points of the scene: distances from a sphere's size to its extent
    tmax = (0.2 * 100.0 ** rand(n)).float()
    return org, dirv, tmax


def _network(seed):
    """Flat fp32 parameters (W1 b1 .. W5 b5): Xavier weights, small biases, lobes told apart by theirs."""
    rng = np.random.default_rng(seed)
    parts = []
    for n, k in LAYERS:
        s = math.sqrt(6.0 / (n + k))
        parts += [rng.uniform(-s, s, n * k), rng.normal(scale=0.5 if n == 40 else 0.05, size=n)]
    return np.concatenate(parts).astype(np.float32)


def _vertices(n, seed):
    """Inputs, directions, radiance weights (a fifth are dark, the rest exponential) and uniforms."""
    rng = np.random.default_rng(seed)
    x = rng.random((n, 7)).astype(np.float32)
    d = rng.normal(size=(n, 3))
    d = (d / np.linalg.norm(d, axis=1, keepdims=True)).astype(np.float32)
    w = rng.exponential(size=n).astype(np.float32)
    w[rng.random(n) < 0.2] = 0.0
    u = np.minimum(rng.random((n, 3)), 1.0 - 2.0 ** -24).astype(np.float32)
    return x, d, w, u


# ---- the cases -----------------------------------------------------------------------------------
def prepare(case, seed):
    kind = case["kind"]
    s = {"case": case}
    if kind in ("guide_grad", "guide_sample"):
        s["guide"] = render.Guide(seed=1)
        s["guide"].set_params(_network(seed))
        s["x"], s["d"], s["w"], s["u"] = _vertices(case["samples"], seed)
        return s
    if kind == "batch":
        sizes = np.random.default_rng(case["images"] * 1000 + case["res"])  # the films are the case's, the scenes the seed's
        items = []
        for i in range(case["images"]):
            n, w, h, k = (int(sizes.integers(lo, hi + 1)) for lo, hi in ((8, case["spheres"]), (32, case["res"]),
                                                                         (32, case["res"]), (8, case["spp"])))
            wl = configs.c1_spheres(w, h, k, seed=seed + i, n_spheres=n)
            items.append((render.GpuScene(wl.scene), wl.camera, k, wl.seed))
        s["batch"] = render.Batch(items, max_depth=16, queue_size=case["queue"])
        return s
    wl = _workload(case, seed)
    if kind == "build":
        s["scene"] = wl.scene
        wl.scene.freeze()
    else:
        s["gscene"] = render.GpuScene(wl.scene)
    if kind in ("trace", "build"):
        s["org"], s["dir"], s["tmax"] = _rays(wl, case["rays"], seed, "cuda")
        return s
    desc = wl.render_desc(integrator=_abi.SPK_INTEGRATOR_DIRECT if case["integrator"] == "direct" else None)
    s["render"] = render.GpuRender(s["gscene"], wl.camera, desc, queue_size=case["queue"])
    if "train_spp" in case:
        s["guide"] = render.Guide(seed=1, train_spp=case["train_spp"])
        s["params"] = _network(seed)
    return s


def run(s):
    case = s["case"]
    kind = case["kind"]
    if kind == "trace":
        if case["any_hit"]:
            return s["gscene"].trace(s["org"], s["dir"], s["tmax"], any_hit=True)[0]
        return s["gscene"].trace(s["org"], s["dir"])
    if kind == "build":
        gs = render.GpuScene(s["scene"], builder="lbvh")
        out = gs.trace(s["org"], s["dir"])
        torch.cuda.current_stream().synchronize()  # the scene is given back while nothing traces it
        gs.close()
        return out
    if kind == "batch":
        s["batch"].run()
        return [s["batch"].film(i) for i in range(case["images"])]
    if kind == "guide_grad":
        loss, grad = s["guide"].grad(s["x"], s["d"], s["w"])
        return np.float32(loss), grad  # the loss is a 32-bit sum, in no fixed order
    if kind == "guide_sample":
        return s["guide"].sample(s["x"], s["u"])
    if "guide" in s:  # a new network, trained online over the pass's first samples
        s["guide"].set_params(s["params"])
        s["render"].set_guide(s["guide"])
    s["render"].run(case["spp"])
    return s["render"].image()


# What a ray needs at the least: a descent of 4-wide nodes (four boxes of three slabs: 24 multiply-adds
# and 22 comparisons a node) and one triangle test.
def _ray_flops(tris):
    return 70.0 * max(1.0, math.log(max(tris, 4), 4)) + 50.0


def _tris(case):
    return 36 if case.get("scene") == "cornell" else 640 * case["spheres"] + 24


def work(case):
    kind = case["kind"]
    if kind == "trace":
        n, t = case["rays"], _tris(case)
        return {"bytes": 32 * n + 36 * t, "flops": n * _ray_flops(t)}
    if kind == "build":
        n, t = case["rays"], _tris(case)
        return {"bytes": 44 * t + 32 * n, "flops": n * _ray_flops(t) + 100.0 * t * math.log2(max(t, 2))}
    if kind == "batch":  # means of the drawn ranges; the film is sums, squares and counts in 64 bits
        px = case["images"] * ((32 + case["res"]) / 2.0) ** 2
        t = 640 * (8 + case["spheres"]) / 2.0
        return {"bytes": 56 * px + 100 * case["images"] * t, "flops": px * (8 + case["spp"]) / 2.0 * 2.0 * _ray_flops(t)}
    if kind == "guide_grad":
        fwd = 2.0 * sum(n * k for n, k in LAYERS)
        return {"bytes": 44 * case["samples"] + 8 * 29480, "flops": case["samples"] * (3.0 * fwd - 2.0 * 64 * 224)}
    if kind == "guide_sample":
        return {"bytes": 56 * case["samples"] + 4 * 29480, "flops": case["samples"] * 2.0 * sum(n * k for n, k in LAYERS)}
    # a render: at least two rays per path (bench.py's sphere field has 2.04), the film read and written,
    # the scene read, and the image written
    px, t = case["width"] * case["height"], _tris(case)
    flops = px * case["spp"] * 2.0 * _ray_flops(t)
    if "train_spp" in case:
        flops += case["train_spp"] * 2.0 ** 18 * 146432.0  # eight steps of 2^18 samples per eight samples per pixel
    return {"bytes": 140 * px + 100 * t, "flops": flops}


# ---- the same in 64 bits -------------------------------------------------------------------------
def _closest_t(verts, org, dirv):
    """Distance to the nearest triangle by testing them all, -1 where there is none."""
    d = _unit(dirv)
    v0, e1, e2 = verts[:, 0], verts[:, 1] - verts[:, 0], verts[:, 2] - verts[:, 0]
    best = torch.full((len(org),), math.inf, dtype=torch.float64, device=org.device)
    step = max(1, 40_000_000 // len(verts))
    dot = lambda a, b: a[..., 0] * b[..., 0] + a[..., 1] * b[..., 1] + a[..., 2] * b[..., 2]  # noqa: E731
    for i in range(0, len(org), step):
        o, w = org[i:i + step, None], d[i:i + step, None]
        p = torch.linalg.cross(w, e2[None])
        det = dot(p, e1)
        tv = o - v0
        u = dot(tv, p) / det
        q = torch.linalg.cross(tv, e1[None].expand_as(tv))
        v = dot(q, w) / det
        t = dot(q, e2) / det
        ok = (det.abs() >= 1e-12) & (u >= 0) & (v >= 0) & (u + v <= 1) & (t > 1e-12)
        best[i:i + step] = torch.where(ok, t, math.inf).amin(dim=1)
    return torch.where(torch.isinf(best), -1.0, best)


def _forward(theta, x):
    """Outputs [n, 8, 5] of the network for inputs x [n, 7]."""
    b = torch.arange(32, dtype=torch.float64, device=x.device) + 0.5
    a = torch.exp(-0.5 * (32.0 * x[:, :, None] - b) ** 2).reshape(len(x), 224)
    at = 0
    for i, (n, k) in enumerate(LAYERS):
        a = a @ theta[at:at + n * k].reshape(n, k).T + theta[at + n * k:at + n * k + n]
        at += n * k + n
        a = torch.relu(a) if i < 4 else a
    return a.reshape(len(x), 8, 5)


def _log_density(o, w):
    mu = o[:, :, 1:4] / torch.sqrt((o[:, :, 1:4] ** 2).sum(-1, keepdim=True).clamp(min=1e-12))
    r = o[:, :, 4].clamp(-4.0, 7.0)
    k = torch.exp(r)
    lobe = r - math.log(2 * math.pi) - torch.log(-torch.expm1(-2.0 * k)) + k * ((mu * w[:, None]).sum(-1) - 1.0)
    return torch.logsumexp(torch.log_softmax(o[:, :, 0], 1) + lobe, 1), mu, k


def exact(case, seed):
    kind = case["kind"]
    dev = "cuda" if torch.cuda.is_available() else "cpu"
    f64 = lambda a: torch.from_numpy(a).to(dev).double()  # noqa: E731
    if kind in ("trace", "build"):
        wl = _workload(case, seed)
        if case.get("any_hit") or case["rays"] * wl.scene.num_tris > 12_000_000_000:
            return None  # whole numbers alone, or too many pairs to test them all
        org, dirv, _ = _rays(wl, case["rays"], seed, "cuda")
        return None, _closest_t(f64(wl.scene.freeze()["verts"]), org.to(dev).double(), dirv.to(dev).double())
    if kind == "guide_grad":
        x, d, w, _ = (f64(a) for a in _vertices(case["samples"], seed))
        theta = f64(_network(seed)).requires_grad_()
        for i in range(0, len(x), 1 << 16):
            part = -(w[i:i + (1 << 16)] * _log_density(_forward(theta, x[i:i + (1 << 16)]), d[i:i + (1 << 16)])[0]).sum()
            (part / len(x)).backward()
        return None, theta.grad
    if kind == "guide_sample":
        x, _, _, u = (f64(a) for a in _vertices(case["samples"], seed))
        o = _forward(f64(_network(seed)), x)
        cdf = torch.cumsum(torch.softmax(o[:, :, 0], 1), 1)
        pick = (u[:, :1] >= cdf).sum(1).clamp(max=7)
        _, mu, k = _log_density(o, u)
        at = torch.arange(len(x), device=dev)
        mu, k = mu[at, pick], k[at, pick]
        cz = (1.0 + torch.log1p((1.0 - u[:, 1]) * torch.expm1(-2.0 * k)) / k).clamp(-1.0, 1.0)
        sz, ph = torch.sqrt(1.0 - cz * cz), 2 * math.pi * u[:, 2]
        sg = torch.where(mu[:, 2] >= 0, 1.0, -1.0).double()
        a = -1.0 / (sg + mu[:, 2])
        b = mu[:, 0] * mu[:, 1] * a
        t1 = torch.stack([1.0 + sg * mu[:, 0] ** 2 * a, sg * b, -sg * mu[:, 0]], 1)
        t2 = torch.stack([b, sg + mu[:, 1] ** 2 * a, -mu[:, 1]], 1)
        w = cz[:, None] * mu + sz[:, None] * (torch.cos(ph)[:, None] * t1 + torch.sin(ph)[:, None] * t2)
        return w, torch.exp(_log_density(o, w)[0])
    # A render decides on 32-bit numbers at every vertex (which triangle, which lobe, whether a path
    # goes on), so its image is a sample of the same estimator in 64 bits, not a rounding of it.
    return None

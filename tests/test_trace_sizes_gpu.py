"""Ray queries at the sizes where the launch is cut differently (rays per wave, chunks per wave): one
ray, the edges of a wave, of the spread over 4,096 waves and of the full grid.  Each call answers its
rays as one large call over all of them does, and a scene of one leaf and an empty one answer too."""
import numpy as np
import pytest

from spica_amd import configs
from spica_amd.scene import Scene, diffuse

pytestmark = pytest.mark.gpu

SIZES = [1, 63, 64, 65, 4095, 4096, 4097, 8193, 16385, 65536, 65537, 131073, 174_763, 524_288, 524_289, 1_048_577]


def _rays(n, spread=6.0):
    import torch

    rng = np.random.default_rng(9)
    org = torch.from_numpy((spread * rng.normal(size=(n, 3))).astype(np.float32)).cuda()
    dirv = torch.from_numpy(rng.normal(size=(n, 3)).astype(np.float32)).cuda()
    tmax = torch.from_numpy(rng.uniform(0.5, 30.0, n).astype(np.float32)).cuda()
    return org, dirv, tmax


@pytest.mark.parametrize("noalloc", [False, True])
def test_sizes_answer_alike(gpu, noalloc):
    import torch

    gs = gpu.GpuScene(configs.c1_spheres(n_spheres=64).scene)
    org, dirv, tmax = _rays(1_700_000)
    p_all, t_all = gs.trace(org, dirv)
    o_all, _ = gs.trace(org, dirv, tmax, any_hit=True)
    assert (p_all >= 0).any() and (p_all < 0).any() and (o_all == 1).any()
    for n in SIZES:
        lo = len(org) - n  # not the slice the large call gives the same waves
        p, t = gs.trace(org[lo:], dirv[lo:], noalloc=noalloc)
        o, _ = gs.trace(org[lo:], dirv[lo:], tmax[lo:], any_hit=True, noalloc=noalloc)
        torch.cuda.synchronize()
        assert torch.equal(p, p_all[lo:]) and torch.equal(t, t_all[lo:]) and torch.equal(o, o_all[lo:]), n
    gs.close()


@pytest.mark.parametrize("tris", [0, 1, 3])
def test_smallest_scenes(gpu, tris):
    import torch

    rng = np.random.default_rng(4)
    v = rng.uniform(-1, 1, size=(tris, 3, 3)).astype(np.float32)
    s = Scene()
    s.add_triangles(v, diffuse((0.5, 0.5, 0.5)))
    gs = gpu.GpuScene(s)
    org, dirv, _ = _rays(5000, 2.0)
    p, t = gs.trace(org, dirv)
    # brute force in float64
    o, d = org.cpu().numpy().astype(np.float64), dirv.cpu().numpy().astype(np.float64)
    d /= np.linalg.norm(d, axis=1, keepdims=True)
    best = np.full(len(o), np.inf)
    for k in range(tris):
        e1, e2 = (v[k, i].astype(np.float64) - v[k, 0] for i in (1, 2))
        pv = np.cross(d, e2)
        det = pv @ e1
        tv = o - v[k, 0]
        u = (tv * pv).sum(1) / det
        q = np.cross(tv, e1)
        w = (q * d).sum(1) / det
        tt = q @ e2 / det
        best = np.where((u >= 0) & (w >= 0) & (u + w <= 1) & (tt > 1e-12) & (tt < best), tt, best)
    hit = np.isfinite(best)
    assert np.array_equal((p >= 0).cpu().numpy(), hit) and (hit.any() or tris == 0)
    assert np.allclose(t.cpu().numpy()[hit], best[hit], rtol=1e-5)
    gs.close()

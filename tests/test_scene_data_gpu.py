"""Scene data formed on the device (triangle records, 4-wide nodes of an LBVH build): pixel means of scenes of one
triangle and of smooth, flat and zero-normal meshes match the oracle's, and both builders give the same film."""
import numpy as np
import pytest

from helpers import zstats
from spica_amd import configs
from spica_amd.scene import Camera, Scene, diffuse, look_at, quad, unit_sphere

pytestmark = pytest.mark.gpu


def _scene(kind):
    s = Scene()
    light = quad((-1, 4, -1), (1, 4, -1), (1, 4, 1), (-1, 4, 1)).reshape(-1, 3, 3)
    if kind in ("back", "front"):  # one emitting triangle, seen from behind (black) or from the front
        t = light[:1] - np.float32([0, 3, 0])
        s.add_triangles((t if kind == "back" else t[:, ::-1]).astype(np.float32), diffuse((0, 0, 0)), radiance=(2, 3, 4))
        return s
    u = unit_sphere(10, 7).reshape(-1, 3, 3)
    nrm = u / np.maximum(np.linalg.norm(u, axis=-1, keepdims=True), 1e-20)
    for i, normals in enumerate((nrm, None, np.zeros_like(nrm))):
        v = u + np.float32([2.3 * (i - 1), 0, 0])
        s.add_triangles(v.astype(np.float32), diffuse((0.7, 0.6, 0.5)),
                        normals=None if normals is None else normals.astype(np.float32))
    s.add_triangles(quad((-5, -1, -5), (-5, -1, 5), (5, -1, 5), (5, -1, -5)).reshape(-1, 3, 3), diffuse((0.5, 0.5, 0.5)))
    s.add_triangles(light, diffuse((0, 0, 0)), radiance=(9, 8, 7))
    return s


@pytest.mark.parametrize("kind", ["back", "front", "smooth"])
def test_film_matches_oracle(gpu, oracle, kind):
    s = _scene(kind)
    cam = Camera(32, 20, look_at((0.3, 2.5, -8), (0, 0.2, 0), (0, 1, 0)), 45.0)
    wl = configs.Workload("scene-data", s, cam, 1024, 4, 0, 11)
    films = []
    for builder in ("sah", "lbvh"):
        gs = gpu.GpuScene(s, builder=builder)
        gr = gpu.GpuRender(gs, cam, wl.render_desc())
        gr.run(1024)
        films.append(gr.film())
        gr.close()
        gs.close()
    assert all(np.array_equal(a, b) for a, b in zip(*films))
    sg, qg, cg = films[0]
    sc, qc, cc, _ = oracle.scene(s).render(cam, wl.render_desc(seed=97), threads=16)
    z, mg, _ = zstats(sg.reshape(-1, 3), qg.reshape(-1, 3), cg.reshape(-1)[:, None], sc, qc, cc[:, None])
    assert (mg.max() > 0) == (sc.max() > 0) == (kind != "back")
    # the pixel criterion of the parity tests: at most 0.5% of channels beyond 3 sigma, none beyond 6
    assert np.mean(np.abs(z) > 3) <= 0.005 and np.abs(z).max() < 6.0, (np.mean(np.abs(z) > 3), np.abs(z).max())

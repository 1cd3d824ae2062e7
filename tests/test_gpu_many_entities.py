"""Scenes with more analytic entities than a block keeps in LDS: closest hits
against the oracle bit for bit, and every engine's image."""
import copy

import numpy as np
import pytest

from oracle.oracle import OracleScene
from prender_amd import generators as G

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def prt():
    from prender_amd import prt as P
    assert P.device_info()["arch"].startswith("gfx950")
    return P


def scene(spheres, planes, mesh, lights=0):
    """The walls of the sphere box (or of the quad box, for none), then spheres and
    rectangles in turn, some of them twice in one place: the lower index wins."""
    d = copy.deepcopy(G.cornell_spheres(width=20, height=16, samples=1) if spheres else
                      G.config2(width=20, height=16, samples=1, level=2))
    rng = np.random.default_rng(5)
    lo, hi = ((10, 5, 20), (90, 70, 120)) if spheres else ((-0.9, 0.1, -0.9), (0.9, 1.9, 0.9))
    size, reach = (1.0, 1.5) if spheres else (0.02, 0.4)
    at = rng.uniform(lo, hi, (spheres + planes + lights, 3))
    for i in range(max(spheres, planes)):
        if i < spheres:
            j = i - 1 if i % 7 == 6 else i
            d.entities.append(G.Sphere(tuple(at[j]), size * (1.0 + j % 3), i % 3))
        if i < planes:
            j = i - 1 if i % 5 == 4 else i
            u, v = rng.normal(size=(2, 3))
            if i % 5 != 4:
                keep = u, v - u * np.dot(u, v) / np.dot(u, u)
            d.entities.append(G.UVPlane(tuple(at[spheres + j]), tuple(reach * keep[0]), tuple(reach * keep[1]), 0))
    if lights:
        d.materials.append(G.Material(color=(0.0, 0.0, 0.0), emission=(8.0, 7.0, 6.0)))
        for p in at[spheres + planes:]:
            d.entities.append(G.Sphere(tuple(p), 0.4 * size, len(d.materials) - 1))
    if mesh:
        v, f = G.displaced_latlong(800, 14.0, (50.0, 14.0, 100.0), 17)
        d.entities.append(G.Polygon(v, f, 0))
    return d


# just above the LDS copy's 16; odd and even counts; no sphere, no rectangle
CASES = [(8, 0, 0, 0), (9, 0, 0, 0), (0, 17, 0, 0), (21, 20, 1, 0), (60, 1, 1, 30)]


@pytest.mark.parametrize("spheres,planes,mesh,lights", CASES)
def test_hits_match_oracle(prt, spheres, planes, mesh, lights):
    d = scene(spheres, planes, mesh, lights)
    rng = np.random.default_rng(6)
    n = 30_011
    lo, hi = ((5, 3, 15), (95, 75, 150)) if spheres else ((-0.95, 0.05, -0.95), (0.95, 1.95, 3.0))
    dirs = rng.normal(size=(n, 3))
    dirs /= np.linalg.norm(dirs, axis=1, keepdims=True)
    rays = G.rays_to_array(rng.uniform(lo, hi, (n, 3)), dirs)
    print(spheres, planes, mesh, lights, flush=True)
    hits, _ = prt.Scene(d).trace(rays)
    ref, _, _ = OracleScene(d).trace(rays)
    assert len(np.unique(ref["entity"])) > 12
    assert np.array_equal(hits["entity"], ref["entity"]) and np.array_equal(hits["t"], ref["t"])


@pytest.mark.parametrize("spheres,planes,mesh,lights", CASES)
@pytest.mark.parametrize("nee", [0, 1])
def test_engines_agree(prt, spheres, planes, mesh, lights, nee):
    d = scene(spheres, planes, mesh, lights)
    d.sampling.next_event_estimation = nee
    print(spheres, planes, mesh, lights, nee, flush=True)
    s = prt.Scene(d)
    a, va, sa = s.render(seed=3, engine=1)
    assert np.isfinite(a).all() and a.max() > 0.0
    for engine in (0, 2, 3):
        b, vb, sb = s.render(seed=3, engine=engine)
        assert np.array_equal(a, b) and np.array_equal(va, vb), engine
        assert sa["shadow_rays"] == sb["shadow_rays"] and sa["extension_rays"] == sb["extension_rays"]

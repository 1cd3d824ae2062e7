"""Traversal stacks beyond the levels kept in LDS, and rays that drop most of
their stack after a hit: meshes of large overlapping triangles, whose nodes have
all their children hit, against the oracle and engine against engine."""
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


def soup(n, size, seed):
    """The triangle box with n random triangles of about `size` in it."""
    d = G.config2(width=24, height=18, samples=2, level=3)
    rng = np.random.default_rng(seed)
    box = next(e for e in d.entities if isinstance(e, G.Polygon))
    lo, hi = box.vertices.min(0), box.vertices.max(0)
    c = rng.uniform(lo + 0.2 * (hi - lo), hi - 0.2 * (hi - lo), (n, 1, 3))
    v = c + rng.normal(size=(n, 3, 3)) * size * (hi - lo) / 4
    d.entities.append(G.Polygon(v.reshape(-1, 3), np.arange(3 * n).reshape(-1, 3), 0))
    return d, lo, hi


@pytest.mark.parametrize("n,size", [(5, 1.0), (300, 1.0), (4000, 0.8), (20000, 0.05)])
def test_deep_stacks(prt, n, size):
    print("triangles", n, flush=True)
    d, lo, hi = soup(n, size, n)
    rng = np.random.default_rng(1)
    org = rng.uniform(lo, hi, (6000, 3))
    dirs = rng.normal(size=(6000, 3))
    dirs[::7, 0] = 0.0  # along an axis plane
    dirs[::49, 1] = 0.0
    dirs /= np.linalg.norm(dirs, axis=1, keepdims=True)
    rays = G.rays_to_array(org, dirs)
    s = prt.Scene(d)
    hits, _ = s.trace(rays)
    ref, _, _ = OracleScene(d).trace(rays, "qbvh")
    assert np.array_equal(hits["entity"], ref["entity"]) and np.array_equal(hits["t"], ref["t"])
    same = hits["prim"] == ref["prim"]  # equal distances within one mesh may take another triangle
    assert same.mean() > 0.999
    assert np.array_equal(hits["u"][same], ref["u"][same]) and np.array_equal(hits["v"][same], ref["v"][same])
    # any hits, and the path kernel's traversal
    a, va, sa = s.render(seed=5, engine=1)
    b, vb, sb = s.render(seed=5, engine=3)
    assert np.isfinite(a).all() and np.array_equal(a, b) and np.array_equal(va, vb)
    assert sa["shadow_rays"] == sb["shadow_rays"] and sa["extension_rays"] == sb["extension_rays"]

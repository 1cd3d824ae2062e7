"""The path kernel (small frames, scenes without light sampling, tails of
depth-synchronous batches) against the depth-synchronous engine, which shares
no scheduling code with it: sums are exact integers, so images, variances and
ray counts are equal bit for bit whatever the grid, the samples a wave holds
and where its light samples and glass branches were traced."""
import numpy as np
import pytest

from prender_amd import generators as G

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def prt():
    from prender_amd import prt as P
    assert P.device_info()["arch"].startswith("gfx950")
    return P


def many_spheres(nee):
    """More analytic entities and materials than a block keeps in LDS."""
    d = G.cornell_spheres(width=24, height=18, samples=2, nee=nee)
    rng = np.random.default_rng(7)
    for i in range(14):
        kind = ("diffuse", "specular", "reflection")[i % 3]
        d.materials.append(G.Material(color=tuple(rng.uniform(0.3, 0.9, 3)), reflection=kind))
        d.entities.append(G.Sphere(tuple(rng.uniform([10, 5, 20], [90, 70, 120])), float(rng.uniform(2, 7)),
                                   len(d.materials) - 1))
    return d


def frame(d, width, height, samples, ss, nee):
    d.camera.width, d.camera.height = width, height
    d.sampling.samples, d.sampling.supersamples, d.sampling.next_event_estimation = samples, ss, nee
    return d


CASES = {
    "one_sample": lambda: frame(G.cornell_spheres(), 1, 1, 1, 1, 0),
    "one_pixel_glass_nee": lambda: frame(G.cornell_spheres(), 1, 1, 5, 3, 1),
    "ragged_glass_nee": lambda: frame(G.cornell_spheres(), 61, 37, 3, 3, 1),
    "many_spheres": lambda: many_spheres(0),
    "many_spheres_nee": lambda: many_spheres(1),
    "box_ragged": lambda: G.config2(width=33, height=17, samples=3, level=3),
    # just below and at the frame size from which three waves share a SIMD
    "box_below_full": lambda: G.config2(width=128, height=127, samples=2, level=3),
    "box_full": lambda: G.config2(width=128, height=128, samples=2, level=3),
    "field_nine_lights": lambda: G.config3(width=64, height=48, samples=3, scale=0.05),
    # depth-synchronous with its tail through the path kernel
    "box_tail": lambda: G.config2(width=301, height=300, samples=3, level=4),
}


@pytest.mark.parametrize("name", list(CASES))
def test_path_kernel_equals_depth_synchronous(prt, name):
    s = prt.Scene(CASES[name]())
    print(name, flush=True)
    a, va, sa = s.render(seed=19, engine=1)
    assert np.isfinite(a).all()
    for engine in (0, 3):
        b, vb, sb = s.render(seed=19, engine=engine)
        assert np.array_equal(a, b) and np.array_equal(va, vb), engine
        assert sa["shadow_rays"] == sb["shadow_rays"] and sa["extension_rays"] == sb["extension_rays"]
        assert sa["pickup_hits"] == sb["pickup_hits"]


def test_path_kernel_vertex_cap(prt):
    s = prt.Scene(G.config2(width=20, height=20, samples=2, level=3))
    a, _, sa = s.render(seed=4, engine=1, max_depth=3)
    b, _, sb = s.render(seed=4, max_depth=3)
    assert np.array_equal(a, b) and sa["truncated_paths"] == sb["truncated_paths"] > 0


def test_split_batch_at_each_register_budget(prt):
    import torch
    scenes = [prt.Scene(d) for d in (G.config1(width=40, height=30, samples=2),
                                     G.config2(width=31, height=29, samples=2, level=3), many_spheres(0))]
    refs = [torch.from_numpy(s.render(seed=6, engine=1)[0]).cuda() for s in scenes]
    for mode in (1, 2):
        for waves in (0, 2, 3, 4):
            out = [torch.zeros_like(r) for r in refs]
            prt.render_batch_device(scenes, [o.data_ptr() for o in out], None,
                                    prt.batch_opts(seed=6, persistent=mode, persist_waves=waves))
            assert all(torch.equal(o, r) for o, r in zip(out, refs)), (mode, waves)

"""The adjoint's recording pass (one traversal of the paths; gradients from the
recorded vertices) at sizes where its records can go wrong: against the oracle's
adjoint, and where a batch has more vertices than records and is replayed."""
import numpy as np
import pytest

from oracle.oracle import OracleScene
from prender_amd import generators as G

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def torch_prt():
    import torch
    from prender_amd import prt as P
    assert P.device_info()["arch"].startswith("gfx950")
    return torch, P


def gradients(torch, prt, d, dimg, albedo=True, light=2, **kw):
    sc = prt.Scene(d)
    nf = d.entities[1].indices.shape[0]
    g = torch.zeros((nf, 3), dtype=torch.float32, device="cuda")
    t = torch.from_numpy(dimg).cuda()
    ge, st = sc.adjoint_device(t.data_ptr(), 1, g.data_ptr() if albedo else None, light, seed=5, **kw)
    return g.cpu().numpy().astype(np.float64), np.asarray(ge), st


# one sample; a partial chunk; several launches' worth of chunks; without light
# sampling.  Same random numbers and paths on both sides: the gradients differ
# by the 2^-32 fixed point of a sample's radiance and the float32 result, the
# bound of the adjoint's other comparisons with the oracle.
@pytest.mark.parametrize("width,height,samples,nee", [(1, 1, 1, 1), (7, 5, 1, 1), (33, 21, 4, 1), (19, 11, 2, 0)])
def test_recorded_gradients_match_oracle(torch_prt, width, height, samples, nee):
    torch, prt = torch_prt
    d = G.config5(width=width, height=height, samples=samples)
    d.sampling.next_event_estimation = nee
    dimg = np.random.default_rng(9).uniform(-1, 1, (height, width, 3)).astype(np.float32)
    print(width, height, samples, nee, flush=True)
    g, ge, _ = gradients(torch, prt, d, dimg)
    ref, ge_ref = OracleScene(d).adjoint(seed=5, dimage=dimg, entity=1, light=2)
    assert np.abs(g - ref).sum() <= 1e-3 * np.abs(ref).sum()
    np.testing.assert_allclose(ge, ge_ref, rtol=1e-3, atol=1e-12)


# batches, one gradient without the other, and paths too long for the records
@pytest.mark.parametrize("depth", [None, 250])
def test_recorded_gradients_in_batches(torch_prt, depth):
    torch, prt = torch_prt
    d = G.config5(width=24, height=20, samples=2)
    if depth:
        d.sampling.depth = d.sampling.depth_limit = depth
    dimg = np.random.default_rng(3).uniform(-1, 1, (20, 24, 3)).astype(np.float32)
    print("depth", depth, flush=True)
    g, ge, st = gradients(torch, prt, d, dimg)
    assert np.isfinite(g).all() and np.abs(g).max() > 0.0
    g7, ge7, st7 = gradients(torch, prt, d, dimg, batch_pixels=101)
    # sums of the same doubles in another order, rounded to float32
    np.testing.assert_allclose(g7, g, rtol=1e-5, atol=1e-9 * np.abs(g).max())
    np.testing.assert_allclose(ge7, ge, rtol=1e-9)
    assert st["shadow_rays"] == st7["shadow_rays"]
    none, ge1, _ = gradients(torch, prt, d, dimg, albedo=False)
    assert not none.any()
    np.testing.assert_allclose(ge1, ge, rtol=1e-9)
    g1, _, _ = gradients(torch, prt, d, dimg, light=-1)
    np.testing.assert_allclose(g1, g, rtol=1e-5, atol=1e-9 * np.abs(g).max())

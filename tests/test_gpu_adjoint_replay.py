"""The adjoint's replay, which a batch with more vertices than records falls back
to, against the oracle's adjoint."""
import numpy as np
import pytest

from oracle.oracle import OracleScene
from prender_amd import generators as G

pytestmark = pytest.mark.gpu


# Paths without Russian roulette run to the box's opening, its light or the vertex
# cap, well past the records there are.  Same random numbers and paths on both
# sides: the gradients differ by the 2^-32 fixed point of a sample's radiance and the
# float32 result, the bound of the adjoint's other comparisons with the oracle.
@pytest.mark.parametrize("width,height,samples,nee,batch", [(24, 20, 1, 1, 0), (24, 20, 1, 1, 101), (23, 17, 2, 0, 0)])
def test_replayed_gradients_match_oracle(width, height, samples, nee, batch):
    import torch
    from prender_amd import prt
    assert prt.device_info()["arch"].startswith("gfx950")
    d = G.config5(width=width, height=height, samples=samples)
    d.sampling.next_event_estimation = nee
    d.sampling.depth = d.sampling.depth_limit = 250
    dimg = np.random.default_rng(9).uniform(-1, 1, (height, width, 3)).astype(np.float32)
    print(width, height, samples, nee, batch, flush=True)
    sc = prt.Scene(d)
    g = torch.zeros((d.entities[1].indices.shape[0], 3), dtype=torch.float32, device="cuda")
    t = torch.from_numpy(dimg).cuda()
    ge, st = sc.adjoint_device(t.data_ptr(), 1, g.data_ptr(), 2, seed=5, batch_pixels=batch)
    # a replay traces every camera ray a second time
    assert st["primary_rays"] == 2 * width * height * d.sampling.supersamples ** 2
    ref, ge_ref = OracleScene(d).adjoint(seed=5, dimage=dimg, entity=1, light=2)
    assert np.abs(ref).sum() > 0.0
    assert np.abs(g.cpu().numpy().astype(np.float64) - ref).sum() <= 1e-3 * np.abs(ref).sum()
    np.testing.assert_allclose(ge, ge_ref, rtol=1e-3, atol=1e-12)

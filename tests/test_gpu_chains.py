"""Markov chains that run each at their own pace against chains stepped
together: a glass sphere that no path can meet (outside the closed box) sends
the same scene's chains step by step.  Splats are integer sums and each chain's
random numbers are its own, so images and counters are equal bit for bit."""
import numpy as np
import pytest

from prender_amd import generators as G

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def prt():
    from prender_amd import prt as P
    assert P.device_info()["arch"].startswith("gfx950")
    return P


def pair(prt, nee, **kw):
    scenes = []
    for glass in (False, True):
        d = G.config2(samples=2, level=3, **kw)
        d.sampling.next_event_estimation = nee
        if glass:
            d.materials.append(G.Material(color=(0.9, 0.9, 0.9), reflection="reflection"))
            d.entities.append(G.Sphere((1.0e4, 1.0e4, 1.0e4), 1.0, len(d.materials) - 1))
        scenes.append(prt.Scene(d))
    return scenes


def same(a, b, keys):
    assert np.isfinite(a[0]).all() and a[0].max() > 0.0
    assert np.array_equal(a[0], b[0])
    for k in keys:
        assert a[1][k] == b[1][k], k


COUNTS = ("camera_samples", "primary_rays", "extension_rays", "shadow_rays", "mlt_proposals", "mlt_accepts")


# one chain; fewer and more than a wave; more chains than a launch's lanes; a
# step past the steps of one launch; vertices past the primary samples
@pytest.mark.parametrize("chains,steps,depths,nee", [(1, 3, 8, 1), (63, 5, 1, 0), (4099, 4, 8, 1), (140001, 2, 3, 1),
                                                     (70, 257, 8, 1)])
def test_chains_at_their_own_pace_equal_chains_in_step(prt, chains, steps, depths, nee):
    a, b = pair(prt, nee, width=37, height=29)
    print(chains, steps, depths, nee, flush=True)
    kw = dict(seed=11, chains=chains, mutations_per_chain=steps, sample_depths=depths)
    same(a.render_mlt(**kw), b.render_mlt(**kw), COUNTS)


@pytest.mark.parametrize("width,mutation", [(5, 3), (90, 4)])
def test_redistribution_chains_at_their_own_pace_equal_chains_in_step(prt, width, mutation):
    a, b = pair(prt, 1, width=width, height=17)
    print(width, mutation, flush=True)
    same(a.render_erpt(seed=5, mutation=float(mutation)), b.render_erpt(seed=5, mutation=float(mutation)), COUNTS)

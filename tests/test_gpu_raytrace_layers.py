"""The traced field stage against rendering the screen first, bit for bit, over
the forms of its layers: one to seven of them (groups of three and the rest),
columns that stay consecutive and ones that skip (magnification), rotated
layers (point by point), windows that leave a layer on either side (the points
outside add nothing), and windows of 16 points and fewer."""
import numpy as np
import pytest

from shwfs import configs, system

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nlayers,pd,nfft,G,theta,edge", [
    (1, 16, 32, 1.0, 0.0, 0), (2, 8, 16, 1.0, 0.0, 0), (3, 13, 32, 1.0, 0.0, 0),
    (4, 16, 32, 1.003, 0.0, 0), (5, 16, 32, 0.97, 0.0, 0), (7, 6, 16, 1.0, 0.0, 0),
    (3, 16, 32, 1.0, 0.1, 0), (3, 16, 32, 1.0, 0.0, 1), (4, 7, 16, 1.02, 0.0, 1),
    (6, 16, 32, 1.0, 0.0, -1), (2, 16, 32, 0.99, -0.3, 1)])
def test_traced_equals_rendered(nlayers, pd, nfft, G, theta, edge):
    c = configs.sh_config(0.2 * 10, 10, pd, 4, nfft, 2, nphot=1000.0)
    c["p_wfs"].G, c["p_wfs"].thetaML = G, theta
    s = system.ShSystem(c)
    n = s.p_geom._n
    rng = np.random.default_rng(10 * nlayers + pd)
    dims = np.full(nlayers, n + (40 if edge == 0 else 3), np.int64)
    z = np.zeros(nlayers, np.float32)
    at = s.sutra.Atmos(s.ctx, nlayers, 0.16, z + 10, dims, np.full(nlayers, 4, np.int64), z, z, z,
                       z, z, 0)
    gs = s.wfs.d_gs
    for k in range(nlayers):
        at.d_screens[k].d_screen.host2device(
            np.asfortranarray(rng.standard_normal((dims[k], dims[k])).astype(np.float32)))
        lo, hi = ((14.0, 26.0), (1.0, 25.0), (-25.0, 0.5))[edge]
        xo, yo = rng.uniform(lo, hi, 2)
        gs.add_layer("atmos", k, float(np.float32(xo)), float(np.float32(np.round(yo))))
    got = []
    for lazy in (True, False):
        gs.lazy_raytrace = lazy
        gs.raytrace(at)
        assert gs.npending == (nlayers if lazy else 0)
        s.comp_image(noise=False)
        s.do_centroids()
        got.append((s.bincube(), s.binimg(), s.intensities(), s.slopes()))
    print("layers %d pd %d G %g theta %g edge %d: nvalid %d" % (nlayers, pd, G, theta, edge,
                                                               s.wfs.nvalid), flush=True)
    for a, b in zip(*got):
        assert np.isfinite(a).all() and np.array_equal(a, b)


@pytest.mark.parametrize("xo,yo", [(3e9, 5.0), (5.0, 3e9), (-3e9, 5.0), (5.0, -3e9), (3e9, 3e9),
                                   (float("inf"), 5.0), (5.0, float("inf"))])
@pytest.mark.parametrize("theta", [0.0, 0.2])
def test_layers_past_the_index_range_add_nothing(xo, yo, theta):
    """A layer shifted further than an int holds: no point falls on it."""
    c = configs.sh_config(0.2 * 10, 10, 16, 4, 32, 2, nphot=1000.0)
    c["p_wfs"].thetaML = theta
    s = system.ShSystem(c)
    n = s.p_geom._n
    dim = n + 60
    z = np.zeros(2, np.float32)
    at = s.sutra.Atmos(s.ctx, 2, 0.16, z + 10, np.full(2, dim, np.int64), np.full(2, 4, np.int64),
                       z, z, z, z, z, 0)
    rng = np.random.default_rng(4)
    for k in range(2):
        at.d_screens[k].d_screen.host2device(
            np.asfortranarray(rng.standard_normal((dim, dim)).astype(np.float32)))
    gs = s.wfs.d_gs
    gs.add_layer("atmos", 0, 30.25, 29.5)
    got = []
    for lazy in (True, False):
        gs.lazy_raytrace = lazy
        gs.raytrace(at)
        s.comp_image(noise=False)
        got.append(s.bincube())
    gs.add_layer("atmos", 1, xo, yo)
    for lazy, want in zip((True, False), got):
        gs.lazy_raytrace = lazy
        gs.raytrace(at)
        s.comp_image(noise=False)
        assert np.isfinite(want).all() and np.array_equal(s.bincube(), want)

"""Correlation maps, maxima and slopes at every spot size (each is a kernel of
its own) and sub-aperture count around a workgroup's four, against the float64
oracle.  A lag sums up to n^2 products in float32: bar 4 n^2 / 2 units of
rounding of the largest lag, and the fit from the device's own map within 2e-5
of the scale."""
import numpy as np
import pytest

import capi
from oracle import corr as oc
from test_gpu_corr import _run, _spots

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("npix,nxsub", [(2, 1), (3, 2), (4, 2), (5, 3), (7, 3), (9, 2), (10, 3),
                                        (11, 1), (13, 2), (14, 3), (15, 2), (16, 4)])
def test_every_spot_size(npix, nxsub):
    lib = capi.load()
    rng = np.random.default_rng(npix)
    pos = [(i * npix, j * npix) for j in range(nxsub) for i in range(nxsub)]
    vx, vy = (np.array([p[k] for p in pos], np.int32) for k in (0, 1))
    img = _spots(rng, npix, nxsub, pos).astype(np.float32).astype(np.float64)
    x = np.arange(npix)
    ref = np.exp(-((x[:, None] - npix // 2) ** 2 + (x[None, :] - npix // 2) ** 2) / 4.0)
    ref = (ref * (1 + 0.1 * rng.random((npix, npix)))).astype(np.float32).astype(np.float64)
    scale, offset = 0.4, npix / 2 - 0.5
    sl, cmap, cmax = _run(lib, img, vx, vy, npix, ref.astype(np.float32), None, 3, 3, offset,
                          scale, None, 0)
    nv, worst = len(pos), 0.0
    for s in range(nv):
        m = oc.corr_map(img[vx[s]:vx[s] + npix, vy[s]:vy[s] + npix], ref)
        got = cmap[s].T
        worst = max(worst, np.abs(got - m).max() / np.abs(m).max())
        fx, fy, imax = oc.fit_map(got.astype(np.float64), npix, offset, scale, 3, 3)
        assert cmax[s] == imax
        assert abs(sl[s] - fx) <= 2e-5 * scale and abs(sl[s + nv] - fy) <= 2e-5 * scale
    print("npix %d nvalid %d: map error %.2e" % (npix, nv, worst), flush=True)
    assert worst < 2 * npix ** 2 * 2.0 ** -24 + 2.0 ** -22

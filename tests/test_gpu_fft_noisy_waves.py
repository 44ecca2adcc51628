"""Noisy FFT frames of few sub-apertures (one wave each): the drawn spots, the
detector image and the flux equal those of the N-lane kernel that a named
workgroup size selects, bit for bit, over both transform sizes, both row
splits, spots of fewer and more than 64 pixels, the general binmap, and
sub-aperture counts around a workgroup's four and the kernels' limit of 2,048;
the slopes to the rounding of their sums (64 float32 terms: 64 units)."""
import numpy as np
import pytest

from conftest import relative_array_error
from shwfs import configs, system

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nx,pd,nfft,nrebin,npix,centro", [
    (2, 8, 16, 2, 8, "cog"), (3, 8, 16, 2, 6, "wcog"), (5, 12, 16, 1, 14, "tcog"),
    (8, 7, 16, 3, 5, "cog"), (4, 16, 32, 4, 8, "wcog"), (9, 24, 32, 2, 10, "tcog"),
    (6, 32, 32, 3, 9, "cog"), (7, 10, 32, 2, 16, "wcog"), (51, 16, 32, 4, 8, "cog"),
    (52, 8, 16, 2, 8, "cog")])
def test_wave_kernel_draws_the_same_frame(nx, pd, nfft, nrebin, npix, centro):
    import sutra
    c = configs.sh_config(0.2 * nx, nx + (nx * pd) % 2, pd, npix, nfft, nrebin, noise=1.5,
                          nphot=3000.0, centroider=centro, thresh=3.0 if centro == "tcog" else 0.0,
                          width=4.0)
    s = system.ShSystem(c)
    s.set_phase(system.make_screens(c, 1)[0])
    slopes = s.rtc.d_control[0].d_centroids
    got = []
    for wg in (64, 0):
        s.wfs.set_wg_size(wg)
        s.wfs.set_noise(1.5, 99)
        for _ in range(2):
            sutra.comp_frame(s.wfs, s.centro, slopes, True)
        got.append((s.bincube(), s.binimg(), s.intensities(), s.slopes()))
    print("nvalid %d" % s.wfs.nvalid, flush=True)
    for a, b in zip(got[0][:3], got[1][:3]):
        assert np.array_equal(a, b)
    assert relative_array_error(got[1][3], got[0][3]) < 64 * 2.0 ** -23

"""The enlarged-grid and convolution kernel at every pair of grids (each its
own instantiation: one or two waves per sub-aperture), windows that fill the
transform and ones that do not, and sub-aperture counts around a workgroup's
four, against the float64 oracle (1e-5 of the largest pixel, the frame's
stated bar)."""
import numpy as np
import pytest

from conftest import relative_array_error
from oracle import wfs as ow
from shwfs import configs, system

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nx,pd,nfft,nrebin,npix,conv", [
    (1, 8, 16, 2, 8, True), (2, 16, 16, 2, 7, True), (3, 5, 16, 3, 8, False),
    (2, 8, 16, 3, 8, True), (2, 12, 16, 4, 15, False), (4, 7, 16, 4, 15, True),
    (3, 16, 32, 4, 8, True), (5, 32, 32, 2, 10, True), (2, 20, 32, 4, 15, False),
    (3, 13, 32, 3, 13, True), (2, 40, 64, 4, 16, True), (3, 64, 64, 3, 9, True)])
def test_frame_matches_oracle(nx, pd, nfft, nrebin, npix, conv):
    c = configs.sh_config(0.3 * nx, nx + (nx * pd) % 2, pd, npix, nfft, nrebin, cobs=0.0,
                          fracsub=0.3, nphot=1000.0, r0=0.2)
    s = system.ShSystem(c)
    w, t = s.p_wfs, s.tables()
    phase = system.make_screens(c, 1)[0]
    s.set_phase(phase)
    s.wfs.set_kernconv(conv)
    s.comp_image(noise=False)
    extra = {}
    if w._Ntot != w._Nfft:
        extra["hrmap"], extra["Ntot"] = w._hrmap, w._Ntot
    if conv:
        extra["ftkernel"] = w._ftkernel
    print("nvalid %d nfft %d ntot %d conv %s" % (w._nvalid, w._Nfft, w._Ntot, conv), flush=True)
    b, inten, img = ow.comp_image(phase, t["pupil"], t["scale"], t["offsets"], t["istart"],
                                  t["jstart"], t["validsubsx"], t["validsubsy"], t["binmap"],
                                  t["fluxPerSub"], t["nphot"], t["pdiam"], t["Nfft"], t["npix"],
                                  t["nxsub"], **extra)
    errs = [relative_array_error(g, r) for g, r in ((s.bincube(), b), (s.binimg(), img),
                                                    (s.intensities(), inten))]
    print("  spots %.2e image %.2e flux %.2e" % tuple(errs), flush=True)
    assert max(errs) < 1e-5

"""Noise-free frames of the FFT method: the split-FP16 products (windows of 5
to 16 points at nfft 16 and 32) against the in-register FFT that a named
workgroup size selects, and both against the float64 oracle, over every form
that the products take: each rebin code, the general binmap (nrebin 3), full
and small windows, one sub-aperture to several workgroups, amplitudes far from
1 and windows with no light.

Bars: each spot is a sum of products rounded to float32, so both forms stay
within 1e-6 of the largest pixel of the oracle (8 units of rounding; measured
2e-7), and the products are not further off than the FFT by more than half of
its error and one unit of rounding."""
import numpy as np
import pytest

from conftest import relative_array_error
from oracle import wfs as ow
from shwfs import configs, system

pytestmark = pytest.mark.gpu

SHAPES = [(2, 8, 16, 2, 8), (9, 7, 16, 1, 10), (6, 16, 16, 3, 5), (12, 5, 16, 4, 4),
          (6, 16, 32, 4, 8), (5, 16, 32, 4, 7), (7, 10, 32, 2, 16), (8, 13, 32, 1, 16),
          (10, 9, 32, 3, 9), (17, 16, 32, 2, 10)]


def _system(nx, pd, nfft, nrebin, npix):
    c = configs.sh_config(0.2 * nx, nx + (nx * pd) % 2, pd, npix, nfft, nrebin, nphot=1000.0)
    s = system.ShSystem(c)
    s.set_phase(system.make_screens(c, 1)[0])
    return s, system.make_screens(c, 1)[0]


def _want(s, phase, pupil):
    t = s.tables()
    return ow.comp_image(phase, pupil, t["scale"], t["offsets"], t["istart"], t["jstart"],
                         t["validsubsx"], t["validsubsy"], t["binmap"], t["fluxPerSub"],
                         t["nphot"], t["pdiam"], t["Nfft"], t["npix"], t["nxsub"])


def _both(s):
    out = []
    for wg in (64, 0):
        s.wfs.set_wg_size(wg)
        s.comp_image(noise=False)
        out.append((s.bincube(), s.binimg(), s.intensities()))
    return out


@pytest.mark.parametrize("nx,pd,nfft,nrebin,npix", SHAPES)
def test_products_match_fft_and_oracle(nx, pd, nfft, nrebin, npix):
    s, phase = _system(nx, pd, nfft, nrebin, npix)
    want = _want(s, phase, s.p_geom._mpupil)
    fft, split = _both(s)
    for name, f, p, w in zip(("spots", "image", "flux"), fft, split, (want[0], want[2], want[1])):
        ef, ep = relative_array_error(f, w), relative_array_error(p, w)
        print("nvalid %d %s: FFT %.2e products %.2e" % (s.wfs.nvalid, name, ef, ep), flush=True)
        assert ef < 1e-6 and ep < 1e-6 and ep <= 1.5 * ef + 1.2e-7


@pytest.mark.parametrize("gain", [1e-6, 3.7, 2.5e4])
def test_products_scale_with_the_amplitude(gain):
    """Amplitudes that fp16 holds only through the per-sub-aperture scale."""
    s, phase = _system(6, 16, 32, 4, 8)
    rng = np.random.default_rng(5)
    pupil = (s.p_geom._mpupil * gain * rng.uniform(0.2, 1.0, s.p_geom._mpupil.shape))
    pupil = np.asfortranarray(pupil.astype(np.float32))
    s.wfs.set_pupil(pupil)
    b, _, _ = _want(s, phase, pupil)
    fft, split = _both(s)
    e = [relative_array_error(x[0], b) for x in (fft, split)]
    print("gain %g: FFT %.2e products %.2e" % (gain, *e), flush=True)
    assert e[0] < 1e-6 and e[1] < 1e-6


def test_dark_and_invalid_windows_match_the_fft():
    s, phase = _system(6, 16, 32, 4, 8)
    w = s.p_wfs
    pupil = np.asfortranarray(s.p_geom._mpupil.copy())
    i, j = w._validpuppixx[0], w._validpuppixy[0]
    pupil[i:i + 16, j:j + 16] = 0.0  # no light
    bad = phase.copy()
    i, j = w._validpuppixx[5], w._validpuppixy[5]
    bad[i + 3, j + 4] = np.nan
    i, j = w._validpuppixx[9], w._validpuppixy[9]
    bad[i + 15, j + 15] = np.inf
    s.wfs.set_pupil(pupil)
    s.set_phase(bad)
    fft, split = _both(s)
    for f, p in zip(fft, split):
        assert np.array_equal(np.isnan(f), np.isnan(p))
    f, p = (x[0].reshape(8, 8, -1, order="F") for x in (fft, split))
    assert np.all(f[:, :, 0] == 0) and np.all(p[:, :, 0] == 0)
    assert np.isnan(p[:, :, 5]).all() and np.isnan(p[:, :, 9]).all()


def test_named_workgroup_size_keeps_the_fft():
    """wg_size 64, 128 and 256 all name the in-register FFT (the same bits);
    the default frame is another computation of the same spots (other bits)."""
    s, _ = _system(8, 16, 32, 4, 8)
    got = []
    for wg in (64, 128, 256, 0):
        s.wfs.set_wg_size(wg)
        s.comp_image(noise=False)
        got.append(s.bincube())
    assert np.array_equal(got[0], got[1]) and np.array_equal(got[0], got[2])
    assert 0.0 < relative_array_error(got[3], got[0]) < 1e-6


@pytest.mark.parametrize("nx,pd,nfft,nrebin,npix,products", [
    (12, 4, 16, 2, 8, False), (12, 5, 16, 2, 8, True), (12, 16, 16, 1, 10, True),
    (12, 8, 16, 3, 5, True), (12, 8, 16, 2, 7, True), (72, 8, 16, 3, 5, True),
    (76, 8, 16, 3, 5, False), (76, 9, 16, 3, 5, True), (76, 8, 16, 2, 8, True),
    (12, 4, 32, 4, 8, False), (12, 5, 32, 4, 8, True), (12, 5, 32, 3, 9, True),
    (12, 16, 32, 2, 11, True), (12, 17, 32, 4, 8, False), (12, 16, 64, 4, 8, False)])
def test_forms_that_take_the_products(nx, pd, nfft, nrebin, npix, products):
    """Which frames are the FFT's own bits, on both sides of each edge: windows
    of 5 and 16 points, and at nfft 16 windows of 8 points with the general
    binmap (nrebin 3; 2x2 binning of 7 pixels starts off the block grid) at 4,096
    sub-apertures (72x72: 4,024; 76x76: 4,488)."""
    s, _ = _system(nx, pd, nfft, nrebin, npix)
    fft, default = _both(s)
    e = relative_array_error(default[0], fft[0])
    print("nvalid %d pd %d nfft %d nrebin %d npix %d: %.1e"
          % (s.wfs.nvalid, pd, nfft, nrebin, npix, e), flush=True)
    assert (0.0 < e < 1e-6) if products else all(np.array_equal(a, b)
                                                 for a, b in zip(fft, default))


@pytest.mark.parametrize("pd,nfft,nrebin,npix,spots", [
    (5, 16, 1, 10, 1.05), (5, 16, 2, 8, 1.05), (8, 16, 2, 8, 1.05), (8, 16, 3, 5, 1.1),
    (16, 16, 2, 8, 1.05), (11, 16, 3, 5, 1.1), (5, 32, 4, 8, 1.05), (8, 32, 3, 9, 1.1),
    (11, 32, 3, 9, 1.1), (16, 32, 2, 12, 1.05), (16, 32, 4, 8, 1.05)])
def test_products_are_no_further_off_than_the_fft(pd, nfft, nrebin, npix, spots):
    """Relative error (2-norm) of spots and flux against the oracle, the mean
    over 16 screens.  The two errors are of independent roundings: their ratio
    spreads by 7 % from screen to screen (some 100 sub-apertures each), 1.8 %
    over 16.  Spots: at most 1.05 times the FFT's, 1.1 with the general binmap
    (0.8 to 1.0 and 0.97 to 1.05 over 32 other screens).  Flux: 0.95 (0.4 to 0.9;
    its mean error, which the table's rounding sets, is most of it)."""
    nx = 12
    c = configs.sh_config(0.2 * nx, nx, pd, npix, nfft, nrebin, nphot=1000.0,
                          seeds=range(1, 17))
    s = system.ShSystem(c)
    err = np.zeros((2, 2))
    for phase in system.make_screens(c):
        s.set_phase(phase)
        want = _want(s, phase, s.p_geom._mpupil)
        for k, got in enumerate(_both(s)):
            for q, (g, w) in enumerate(((got[0], want[0]), (got[2], want[1]))):
                err[k, q] += np.linalg.norm(g.astype(np.float64) - w) / np.linalg.norm(w) / 16
    print("pd %d nfft %d nrebin %d: spots %.3e %.3e flux %.3e %.3e"
          % (pd, nfft, nrebin, err[0, 0], err[1, 0], err[0, 1], err[1, 1]), flush=True)
    assert err[1, 0] <= spots * err[0, 0] and err[1, 1] <= 0.95 * err[0, 1]

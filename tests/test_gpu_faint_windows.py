"""Windows of very small amplitude on the methods whose fields carry a
power-of-two scale (the FFT method's split-FP16 products and FP16): the scale
may pass a float's exponent range, the results may not.  Alone and in a batch,
whole windows and the paired 8-point ones.

Spots are normalised to the sub-aperture's flux, so they are the oracle's at
every amplitude: 1e-6 of the largest pixel for the products (8 units of
rounding) and 1e-3 for FP16 operands.  An amplitude of 5e-39 reaches the
largest field factor; it is subnormal, a multiple of 2^-149, which rounds the
field 2.3 times as coarsely: 3e-6.  The raw flux goes with the amplitude
squared: 1e-6 and 1e-3 of it where a float holds it (1e-17 and 1e-20), below
the smallest normal float past that."""
import numpy as np
import pytest

from conftest import relative_array_error
from oracle import wfs as ow
from shwfs import configs, system

pytestmark = pytest.mark.gpu

FFT, FP16 = 0, 2


@pytest.mark.parametrize("gain", [1e-17, 1e-20, 1e-30, 5e-39])
@pytest.mark.parametrize("pd,nfft,nrebin,npix", [(16, 32, 4, 8), (8, 16, 2, 8), (13, 32, 3, 9)])
@pytest.mark.parametrize("method", [FFT, FP16])
def test_faint_windows(method, pd, nfft, nrebin, npix, gain):
    s = system.ShSystem(configs.sh_config(1.6, 8, pd, npix, nfft, nrebin, nphot=1000.0),
                        method=method)
    phase = system.make_screens(s.cfg, 1)[0]
    s.set_phase(phase)
    pupil = np.asfortranarray((s.p_geom._mpupil * gain).astype(np.float32))
    s.wfs.set_pupil(pupil)
    t = s.tables()
    spots, flux, _ = ow.comp_image(phase, pupil, t["scale"], t["offsets"], t["istart"],
                                   t["jstart"], t["validsubsx"], t["validsubsy"], t["binmap"],
                                   t["fluxPerSub"], t["nphot"], t["pdiam"], t["Nfft"], t["npix"],
                                   t["nxsub"])
    batch = s.sutra.WfsBatch(s.ctx, [s.wfs], [s.centro], False)
    batch.set_tiles([method], [0])
    bar = 1e-3 if method == FP16 else 3e-6 if gain < 1e-37 else 1e-6
    frames = [("alone", lambda: s.comp_image(noise=False)), ("batch", batch.launch)]
    if method == FFT and nrebin == 3 and gain < 1e-20:
        frames.pop()  # a general binmap in a batch takes the FFT, whose |F|^2 is 0 there
    for name, frame in frames:
        frame()
        es = relative_array_error(s.bincube(), spots)
        f = s.intensities().astype(np.float64)
        ef = relative_array_error(f, flux) if gain >= 1e-20 else np.abs(f).max()
        print("method %d pd %d gain %g %s: spots %.1e flux %.1e" % (method, pd, gain, name, es, ef),
              flush=True)
        assert es < bar
        assert ef < bar if gain >= 1e-20 else ef < 1e-38

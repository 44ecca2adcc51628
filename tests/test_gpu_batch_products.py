"""Batches of the FFT method at their default tiles (split 0), noise-free: the
same-kind kernel and the registered group kernel run the split-FP16 products
of the frame alone; every other batch, a named workgroup size and a batch with
a noisy member run the in-register FFT that workgroup size 64 names.  Each
route is told by its bits: spots and image equal the frame alone of the same
computation bit for bit, and the other computation's only to 1e-6 of the
largest pixel.  Moments of the products are float64 sums, in one order for
spots of up to 64 pixels (slopes equal bit for bit) and in two for larger ones:
one unit of rounding of a centroid of up to 16 pixels, 2^-20 pixels, against
slopes of at least half a pixel: 2e-6.  Everything within 1e-5 of the float64
oracle."""
import numpy as np
import pytest

from conftest import relative_array_error
from oracle import centroid as oc
from oracle import wfs as ow
from shwfs import configs, system

pytestmark = pytest.mark.gpu


def _cfg(nx, pd, nfft, nrebin, npix, centroider="cog", seed=1):
    nx += (nx * pd) % 2
    return configs.sh_config(0.2 * nx, nx, pd, npix, nfft, nrebin, nphot=1000.0,
                             centroider=centroider, thresh=20.0 if centroider == "tcog" else 0.0,
                             width=4.0 if centroider == "wcog" else None, seeds=[seed])


def _batch(cfgs, noise=False):
    bs = system.BatchSystem(cfgs, noise=noise)
    bs.set_phases([system.make_screens(c, 1)[0] for c in cfgs])
    bs.batch.set_tiles([0] * len(cfgs), [0] * len(cfgs))
    return bs


def _out(bs):
    bs.batch.launch()
    return [(s.bincube(), s.binimg(), bs.slopes(i)) for i, s in enumerate(bs.systems)]


def _alone(s, wg):
    s.wfs.set_wg_size(wg)
    s.sutra.comp_frame(s.wfs, s.centro, s.rtc.d_control[0].d_centroids, False)
    s.wfs.set_wg_size(0)
    return s.bincube(), s.binimg(), s.slopes()


def _check_oracle(s, got):
    t, w, c = s.tables(), s.p_wfs, s.centro
    phase = system.make_screens(s.cfg, 1)[0]
    spots, _, img = ow.comp_image(phase, t["pupil"], t["scale"], t["offsets"], t["istart"],
                                  t["jstart"], t["validsubsx"], t["validsubsy"], t["binmap"],
                                  t["fluxPerSub"], t["nphot"], t["pdiam"], t["Nfft"], t["npix"],
                                  t["nxsub"])
    assert relative_array_error(got[0], spots) < 1e-5
    args = (img, w._validsubsx, w._validsubsy, w.npix)
    kind = s.cfg["p_centroider"].type
    if kind == "cog":
        sl = oc.cog(*args, c.offset, c.scale)[0]
    elif kind == "tcog":
        sl = oc.tcog(*args, c.offset, c.scale, 20.0)[0]
    else:
        wts = np.array(c.d_weights).reshape(w.npix, w.npix, -1, order="F")
        sl = oc.wcog(*args, c.offset, c.scale, wts)[0]
    assert relative_array_error(got[2], sl) < 1e-5


# (windows, transform, binning, pixels): each register binning, full, partial
# and paired windows (products in the batch); the general binmap (nrebin 3, and
# blocks off the rebin grid), whose frames alone take the products
@pytest.mark.parametrize("pd,nfft,nrebin,npix,products", [
    (7, 16, 1, 10, True), (8, 16, 2, 8, True), (7, 16, 4, 4, True), (13, 16, 2, 8, True),
    (16, 16, 4, 4, True), (5, 32, 2, 10, True), (8, 32, 4, 8, True), (13, 32, 1, 12, True),
    (16, 32, 4, 8, True), (16, 32, 2, 12, True), (13, 16, 3, 5, False), (13, 16, 2, 7, False),
    (16, 32, 4, 7, False), (16, 32, 3, 9, False)])
@pytest.mark.parametrize("centroider", ["cog", "tcog", "wcog"])
def test_same_kind(pd, nfft, nrebin, npix, products, centroider):
    cfgs = [_cfg(nx, pd, nfft, nrebin, npix, centroider, seed)
            for seed, nx in enumerate((9, 2, 14), 1)]
    bs = _batch(cfgs)
    for grid, remap in ((0, 0), (64, 1)):
        bs.batch.set_tiles([0] * 3, [0] * 3, grid, remap)
        got = _out(bs)
        for s, g in zip(bs.systems, got):
            same = _alone(s, 0 if products else 64)
            other = _alone(s, 64 if products else 0)
            e = [relative_array_error(a, b) for a, b in zip(g, same)]
            print("nvalid %d grid %d: spots %.1e image %.1e slopes %.1e" % (s.wfs.nvalid, grid, *e),
                  flush=True)
            assert e[:2] == [0.0, 0.0]
            assert e[2] <= (0.0 if npix <= 8 else 2e-6)
            assert 0.0 < relative_array_error(g[0], other[0]) < 1e-6
            _check_oracle(s, g)


MIXED = {
    "nfft 64 beside": [(12, 16, 32, 4, 8), (6, 32, 64, 4, 16)],
    "24-point windows beside": [(12, 16, 32, 4, 8), (10, 24, 32, 4, 8)],
    "two binnings": [(12, 16, 32, 4, 8), (12, 16, 32, 3, 9)],
    "two transforms": [(12, 16, 32, 4, 8), (13, 8, 16, 2, 8)],
    "three kinds, other windows": [(12, 13, 32, 4, 8), (13, 8, 16, 2, 8), (6, 32, 64, 4, 16)],
}


@pytest.mark.parametrize("name", MIXED)
def test_mixed_batches_take_the_fft(name):
    bs = _batch([_cfg(*shape, seed=k + 1) for k, shape in enumerate(MIXED[name])])
    n = len(bs.systems)
    for grid, remap in ((0, 0), (64, 1)):
        bs.batch.set_tiles([0] * n, [0] * n, grid, remap)
        for s, g in zip(bs.systems, _out(bs)):
            fft, default = _alone(s, 64), _alone(s, 0)
            assert relative_array_error(g[0], fft[0]) == 0.0
            assert relative_array_error(g[1], fft[1]) == 0.0
            assert relative_array_error(g[0], default[0]) < 1e-6
            _check_oracle(s, g)


def test_named_workgroup_size_and_noisy_member_take_the_fft():
    cfgs = [_cfg(9, 16, 32, 4, 8, seed=k + 1) for k in range(2)]
    bs = _batch(cfgs)
    for s in bs.systems:
        s.wfs.set_wg_size(256)
    bs.batch = bs.sutra.WfsBatch(bs.systems[0].ctx, [s.wfs for s in bs.systems],
                                 [s.centro for s in bs.systems], False)
    for s, g in zip(bs.systems, _out(bs)):
        assert relative_array_error(g[0], _alone(s, 64)[0]) == 0.0
    # one noisy WFS: the other one's spots are the FFT's too
    bs.systems[1].wfs.set_noise(0.5, 77)
    bs.batch = bs.sutra.WfsBatch(bs.systems[0].ctx, [s.wfs for s in bs.systems],
                                 [s.centro for s in bs.systems], True)
    g, s = _out(bs)[0], bs.systems[0]
    assert relative_array_error(g[0], _alone(s, 64)[0]) == 0.0
    assert 0.0 < relative_array_error(g[0], _alone(s, 0)[0]) < 1e-6


@pytest.mark.parametrize("pd,nfft,nrebin,npix", [(8, 16, 2, 8), (16, 32, 4, 8), (13, 32, 3, 9)])
def test_noisy_fft_batch_against_the_frame_alone(pd, nfft, nrebin, npix):
    """The same draws: spots and image equal bit for bit.  Alone the frame runs
    one wave per sub-aperture and sums its float moments over 64 lanes, in the
    batch over nfft: a few units of rounding of centroids of up to 9 pixels,
    5e-6 of the largest slope."""
    cfgs = [_cfg(nx, pd, nfft, nrebin, npix, seed=nx) for nx in (9, 14)]
    bs = _batch(cfgs)
    for k, s in enumerate(bs.systems):
        s.wfs.set_noise(0.5, 77 + k)
    bs.batch = bs.sutra.WfsBatch(bs.systems[0].ctx, [s.wfs for s in bs.systems],
                                 [s.centro for s in bs.systems], True)
    bs.batch.set_frame(0)
    got = _out(bs)
    for k, s in enumerate(bs.systems):
        s.wfs.set_noise(0.5, 77 + k)  # call counter 0
        s.sutra.comp_frame(s.wfs, s.centro, s.rtc.d_control[0].d_centroids, True)
        e = [relative_array_error(a, b)
             for a, b in zip(got[k], (s.bincube(), s.binimg(), s.slopes()))]
        print("nvalid %d: spots %.1e image %.1e slopes %.1e" % (s.wfs.nvalid, *e), flush=True)
        assert e[:2] == [0.0, 0.0] and e[2] < 5e-6

"""Field stop at every transform length (16 to 4096: each count of radix
passes and of lines per workgroup), with pupils that do not fill the last
workgroup of rows and that fill the whole grid, against the float64 oracle.
The bar is the transforms' rounding: 2 log2(n) float32 steps on the field's
largest value, with the factor 4 of a worst case over n^2 points."""
import numpy as np
import pytest

import capi
from oracle import wfs as ow

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,npup", [(16, 16), (16, 9), (32, 21), (64, 64), (64, 37), (128, 101),
                                    (256, 256), (256, 193), (512, 311), (1024, 1), (1024, 645),
                                    (2048, 1030), (4096, 1283)])
def test_every_length_matches_oracle(n, npup):
    import torch
    lib = capi.load()
    rng = np.random.default_rng(n + npup)
    phase = (2.0 * rng.standard_normal((npup, npup))).astype(np.float32)
    pupil = (0.25 + rng.random((npup, npup))).astype(np.float32)
    k = np.minimum(np.arange(n), n - np.arange(n))  # distance to the zero frequency
    mask = (np.maximum(k[:, None], 1.5 * k[None, :]) < 0.3 * n).astype(np.float32)
    scale = np.float32(2 * np.pi / 0.6)
    t = lambda a: torch.tensor(np.ascontiguousarray(a.T.ravel()), device="cuda")  # x fastest
    d = [t(phase), t(pupil), t(mask)]
    work = torch.zeros(2 * n * npup, dtype=torch.float32, device="cuda")
    oph = torch.zeros(npup * npup, dtype=torch.float32, device="cuda")
    oam = torch.zeros_like(oph)
    print("field stop n=%d npup=%d" % (n, npup), flush=True)
    rc = lib.shwfs_field_stop(capi.ptr(d[0]), capi.ptr(d[1]), npup, float(scale), capi.ptr(d[2]),
                              n, capi.ptr(work), capi.ptr(oph), capi.ptr(oam), None)
    assert rc == 0, capi.last_error(lib)
    torch.cuda.synchronize()
    a = oam.cpu().numpy().astype(np.float64).reshape(npup, npup).T
    p = oph.cpu().numpy().astype(np.float64).reshape(npup, npup).T
    want = ow.field_stop(phase, pupil, float(scale), mask)
    err = np.abs(a * np.exp(1j * float(scale) * p) - want).max() / np.abs(want).max()
    bar = 4 * 2 * np.log2(n) * 2.0 ** -24 + 4 * 2.0 ** -22  # and the output angle's rounding
    print("  error %.2e (bar %.2e)" % (err, bar), flush=True)
    assert err < bar


@pytest.mark.parametrize("n,npup", [(256, 193), (512, 311), (1024, 645), (2048, 1030),
                                    (4096, 1283)])
def test_mean_energy_is_kept(n, npup):
    """An all-pass stop gives the field back: the mean of its squared amplitude
    over tens of thousands of points, where random roundings cancel, keeps what
    the rounded twiddles lose or the output scale gives back.  Half a unit of
    that scale on the amplitude, 2 x 2^-24, and a quarter of that for the
    twiddles between the passes."""
    import torch
    lib = capi.load()
    rng = np.random.default_rng(n)
    phase = (2.0 * rng.standard_normal((npup, npup))).astype(np.float32)
    t = lambda a: torch.tensor(np.ascontiguousarray(a.T.ravel()), device="cuda")
    d = [t(phase), t(np.ones((npup, npup), np.float32)), t(np.ones((n, n), np.float32))]
    work = torch.zeros(2 * n * npup, dtype=torch.float32, device="cuda")
    oph = torch.zeros(npup * npup, dtype=torch.float32, device="cuda")
    oam = torch.zeros_like(oph)
    print("all-pass n=%d npup=%d" % (n, npup), flush=True)
    rc = lib.shwfs_field_stop(capi.ptr(d[0]), capi.ptr(d[1]), npup, 10.0, capi.ptr(d[2]), n,
                              capi.ptr(work), capi.ptr(oph), capi.ptr(oam), None)
    assert rc == 0, capi.last_error(lib)
    torch.cuda.synchronize()
    gain = float((oam.double() ** 2).mean()) - 1.0
    print("  energy %.2e" % gain, flush=True)
    assert abs(gain) < 1.25 * 2.0 ** -23

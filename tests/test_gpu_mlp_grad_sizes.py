"""Loss and gradient of the learned centroider at the sizes where its launch
changes: fewer samples than one wave's, a step's remainder, one and several
steps per workgroup, gradients added by atomics (up to 32 workgroups of 128
samples) and through partial sums, gathered samples, and both again with the
samples' values spread widely; against the float64 oracle on bf16-rounded
inputs and weights.  The remaining differences are the roundings of H1, dZ2
and dZ1 to bf16 (2^-9 each, random over the samples): a bar of 4 x 2^-9 of
the gradient's norm, and of 2^-9 for the loss."""
import numpy as np
import pytest

from oracle import mlp as om

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,gather", [(1, False), (15, True), (127, False), (128, True),
                                      (129, False), (4096, True), (4097, False), (33000, True),
                                      (70001, False)])
def test_gradient_sizes(n, gather):
    import ctypes as C

    import capi
    import torch
    lib = capi.load()
    rng = np.random.default_rng(n)
    p = np.concatenate([(rng.standard_normal(s) * (1 / np.sqrt(s[-1]) if len(s) == 2 else 0.1)).ravel()
                        for _, s in om.SHAPES]).astype(np.float32)
    x = rng.gamma(0.3, 2.0, (n, 64)).astype(np.float32)
    t = rng.uniform(-1, 1, (n, 2)).astype(np.float32)
    order = rng.permutation(n) if gather else np.arange(n)
    dev = lambda a: torch.from_numpy(np.ascontiguousarray(a)).cuda()
    d_p, d_t, d_x = dev(p), dev(t), dev(x)
    d_i = dev(order.astype(np.int32)) if gather else None
    lib.shwfs_mlp_work_bytes.restype = C.c_size_t
    work = torch.zeros(lib.shwfs_mlp_work_bytes(), dtype=torch.uint8, device="cuda")
    grad = torch.full((om.NPARAM,), 7.0, device="cuda")
    loss = torch.full((1,), 7.0, device="cuda")
    lib.shwfs_mlp_loss_grad.argtypes = [C.c_void_p] * 5 + [C.c_int64, C.c_float, C.c_float] + \
        [C.c_void_p] * 3
    print("loss_grad n=%d gather=%s" % (n, gather), flush=True)
    for _ in range(2):  # the second call starts from the first one's buffers
        rc = lib.shwfs_mlp_loss_grad(capi.ptr(d_p), capi.ptr(work), capi.ptr(d_x), capi.ptr(d_t),
                                     capi.ptr(d_i), n, 0.125, 2.0, capi.ptr(grad), capi.ptr(loss),
                                     None)
        assert rc == 0, capi.last_error(lib)
    torch.cuda.synchronize()
    pr = p.astype(np.float64)
    w = om.unpack(pr)
    w["W1"], w["W2"] = om.bf16_round(w["W1"]), om.bf16_round(w["W2"])
    want_l, want_g = om.loss_grad(om.pack(w), om.bf16_round(0.125 * x), 2.0 * t.astype(np.float64))
    g = grad.cpu().numpy().astype(np.float64)
    eg = np.linalg.norm(g - want_g) / np.linalg.norm(want_g)
    el = abs(float(loss) - want_l) / want_l
    print("  gradient %.2e loss %.2e" % (eg, el), flush=True)
    assert eg < 4 * 2.0 ** -9 and el < 2.0 ** -9

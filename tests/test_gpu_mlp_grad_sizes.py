"""Loss and gradient of the learned centroider at the sizes where its launch
changes: fewer samples than one wave's, a step's remainder, one and several
steps per workgroup (up to 256 of them take 128 samples a step), gathered
samples, gradients added by atomics and through partial sums (a d_part and more
than 64 workgroups); against the float64 oracle on bf16-rounded inputs and weights.

The first and the last sample of the last step and one of each later step of a
workgroup have targets 100 times the others', so that each is a large part of
the gradient: one of them left out moves every block by 0.9 % or more.  The
remaining differences are the roundings of H1, dZ2 and dZ1 to bf16 (2^-9 each):
a bar of 4 x 2^-9 of the norm of each of the six blocks, and of 2^-9 for the
loss."""
import numpy as np
import pytest

from oracle import mlp as om

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,gather", [(1, False), (15, True), (127, False), (128, True),
                                      (129, False), (4096, True), (4097, False), (33000, True),
                                      (70001, False)])
@pytest.mark.parametrize("part", [False, True])
def test_gradient_sizes(n, gather, part):
    import ctypes as C

    import capi
    import torch
    lib = capi.load()
    rng = np.random.default_rng(n)
    p = np.concatenate([(rng.standard_normal(s) * (1 / np.sqrt(s[-1]) if len(s) == 2 else 0.1)).ravel()
                        for _, s in om.SHAPES]).astype(np.float32)
    x = rng.gamma(0.3, 2.0, (n, 64)).astype(np.float32)
    t = rng.uniform(-1, 1, (n, 2)).astype(np.float32)
    heavy = np.zeros(n, bool)
    heavy[[n - 1, n - (n % 128 or 128)]] = True  # last step: its last and first sample
    heavy[128 * 256 + 37::128] = True  # a workgroup's steps after its first
    t[heavy] *= 100.0
    order = rng.permutation(n) if gather else np.arange(n)
    dev = lambda a: torch.from_numpy(np.ascontiguousarray(a)).cuda()
    d_p, d_t, d_x = dev(p), dev(t), dev(x)
    d_i = dev(order.astype(np.int32)) if gather else None
    lib.shwfs_mlp_work_bytes.restype = C.c_size_t
    work = torch.zeros(lib.shwfs_mlp_work_bytes(), dtype=torch.uint8, device="cuda")
    grad = torch.full((om.NPARAM,), 7.0, device="cuda")
    loss = torch.full((1,), 7.0, device="cuda")
    lib.shwfs_mlp_part_bytes.restype = C.c_size_t
    d_part = torch.full((lib.shwfs_mlp_part_bytes() // 4,), 7.0, device="cuda") if part else None
    lib.shwfs_mlp_loss_grad_part.argtypes = [C.c_void_p] * 6 + [C.c_int64, C.c_float, C.c_float] + \
        [C.c_void_p] * 3
    print("loss_grad n=%d gather=%s part=%s" % (n, gather, part), flush=True)
    for _ in range(2):  # the second call starts from the first one's buffers
        rc = lib.shwfs_mlp_loss_grad_part(capi.ptr(d_p), capi.ptr(work), capi.ptr(d_part),
                                          capi.ptr(d_x), capi.ptr(d_t), capi.ptr(d_i), n, 0.125,
                                          2.0, capi.ptr(grad), capi.ptr(loss), None)
        assert rc == 0, capi.last_error(lib)
    torch.cuda.synchronize()
    pr = p.astype(np.float64)
    w = om.unpack(pr)
    w["W1"], w["W2"] = om.bf16_round(w["W1"]), om.bf16_round(w["W2"])
    want_l, want_g = om.loss_grad(om.pack(w), om.bf16_round(0.125 * x), 2.0 * t.astype(np.float64))
    got, want = om.unpack(grad.cpu().numpy().astype(np.float64)), om.unpack(want_g)
    eg = {k: np.linalg.norm(got[k] - want[k]) / np.linalg.norm(want[k]) for k in want}
    el = abs(float(loss) - want_l) / want_l
    print("  gradient %s loss %.2e" % (" ".join("%s %.2e" % i for i in eg.items()), el), flush=True)
    assert max(eg.values()) < 4 * 2.0 ** -9 and el < 2.0 ** -9


def test_work_area_depends_on_the_parameters_alone():
    """What calls leave in d_work: the inference copies stay as they are under
    loss_grad, and no sample reaches the area, so that calls with the same
    parameters may share it (here: inference and gradients of two sizes on
    three streams, against the same calls one after the other; the gradients'
    float sums differ in order: 1e-5 of the norm)."""
    import ctypes as C

    import capi
    import torch
    lib = capi.load()
    lib.shwfs_mlp_work_bytes.restype = C.c_size_t
    vp = C.c_void_p
    lib.shwfs_mlp_loss_grad.argtypes = [vp] * 5 + [C.c_int64, C.c_float, C.c_float] + [vp] * 3
    lib.shwfs_mlp_forward.argtypes = [vp] * 3 + [C.c_int64, C.c_float, vp, vp]
    assert lib.shwfs_mlp_work_bytes() < 1 << 18
    rng = np.random.default_rng(11)
    dev = lambda a: torch.from_numpy(np.ascontiguousarray(a, np.float32)).cuda()
    p = dev(np.concatenate([(rng.standard_normal(s) / np.sqrt(s[-1])).ravel()
                            for _, s in om.SHAPES]))
    work = torch.zeros(lib.shwfs_mlp_work_bytes(), dtype=torch.uint8, device="cuda")
    sets = [(dev(rng.gamma(0.3, 2.0, (n, 64))), dev(rng.uniform(-1, 1, (n, 2))), n)
            for n in (40000, 9000)]
    outs = [(torch.zeros(om.NPARAM, device="cuda"), torch.zeros(1, device="cuda")) for _ in sets]
    y = torch.zeros(9000, 2, device="cuda")

    def grad(k, stream):
        x, t, n = sets[k]
        assert lib.shwfs_mlp_loss_grad(capi.ptr(p), capi.ptr(work), capi.ptr(x), capi.ptr(t), None,
                                       n, 0.125, 2.0, capi.ptr(outs[k][0]), capi.ptr(outs[k][1]),
                                       stream) == 0, capi.last_error(lib)

    def forward(stream):
        assert lib.shwfs_mlp_forward(capi.ptr(p), capi.ptr(work), capi.ptr(sets[1][0]), 9000, 0.125,
                                     capi.ptr(y), stream) == 0, capi.last_error(lib)

    forward(None)
    torch.cuda.synchronize()
    want_y, copies = y.clone(), work.clone()
    inference = 2 * (om.NIN * om.NH + om.NH * om.NH)  # bf16 W1 and W2
    left, want = [], []
    for k in range(2):
        grad(k, None)
        torch.cuda.synchronize()
        left.append(work.clone())
        want.append([o.clone() for o in outs[k]])
    assert torch.equal(left[0][:inference], copies[:inference])
    assert torch.equal(left[0], left[1])
    streams = [torch.cuda.Stream() for _ in range(3)]
    for _ in range(5):
        for k in range(2):
            grad(k, streams[k].cuda_stream)
        forward(streams[2].cuda_stream)
    torch.cuda.synchronize()
    assert torch.equal(y, want_y)
    for (g, l), (wg, wl) in zip(outs, want):
        assert float((g - wg).norm() / wg.norm()) < 1e-5 and abs(float(l - wl) / float(wl)) < 1e-5

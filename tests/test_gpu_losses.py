"""Cross-entropy parity (metrics_losses.c:28-125, losses.asm:315-613).

label_smoothing_ce_forward / _backward / _fused against the oracle's
restatement (itself bit-exact against the reference's own C, see
tests/test_oracle_losses.py) and, where the reference build travelled with
the tree, against that C directly.  The loss is a sum over rows and classes
accumulated here in a fixed tree instead of the reference's index order:
|g - r| <= 1e-12 * sum|terms| / B.  Gradients: 1e-12 relative + 2e-15 / B
absolute (softmax - target cancels).  neural_cross_entropy_loss: f64 against
the oracle (same bound), f32 against the fp64 closed form at 2e-6 relative
+ 2e-7 absolute (p_target is rounded to float, as in the reference; near 1 that
rounding is absolute in the loss; the reference's sequential float sums are
reported, not gated).
"""

import ctypes
import math

import numpy as np
import pytest

from conftest import GPU, rel_close, same_bits

pytestmark = GPU


def _case(b, k, seed, special=False):
    rng = np.random.default_rng(seed)
    x = rng.normal(0, 3, (b, k))
    t = rng.integers(0, k, b).astype(np.int64)
    if special and b >= 5 and k >= 4:
        x[0, 1] = np.inf
        x[1, 2] = -np.inf
        x[2, 0] = np.nan
        x[3, k - 1] = np.nan
        x[4, :] = -np.inf
    return x, t


def _bound(x, t, a):
    """sum over rows/classes of |st * log_soft| / B, the scale of the loss sum."""
    b, k = x.shape
    m = np.max(np.where(np.isnan(x), -np.inf, x), axis=1, keepdims=True)
    with np.errstate(all="ignore"):
        lsm = (x - m) - np.log(np.exp(x - m).sum(axis=1, keepdims=True))
    st = np.full((b, k), a / k)
    st[np.arange(b), t] += 1 - a
    with np.errstate(all="ignore"):
        v = np.abs(st * lsm)
    return float(np.nansum(np.where(np.isfinite(v), v, 0))) / b


def _ls_gpu(pn, x, t, a, mode):
    lib = pn.core._lib
    b, k = x.shape
    loss = ctypes.c_double()
    g = np.full((b, k), np.nan)
    if mode == "fwd":
        rc = lib.label_smoothing_ce_forward(x.ctypes.data, t.ctypes.data, b, k, a, ctypes.byref(loss))
    elif mode == "bwd":
        rc = lib.label_smoothing_ce_backward(x.ctypes.data, t.ctypes.data, b, k, a, g.ctypes.data)
    else:
        rc = lib.label_smoothing_ce_fused(x.ctypes.data, t.ctypes.data, b, k, a, ctypes.byref(loss), g.ctypes.data)
    return rc, loss.value, g


def _loss_close(got, want, bound, tol=1e-12):
    if math.isnan(want):
        assert math.isnan(got)
    elif math.isinf(want):
        assert got == want
    else:
        assert abs(got - want) <= tol * bound + 1e-300, (got, want, bound)


@pytest.mark.parametrize("b,k", [(1, 1), (3, 5), (17, 10), (64, 1000), (5, 4096), (300, 2049), (1024, 64)])
@pytest.mark.parametrize("a", [0.0, 0.1, 1.0])
def test_ls_ce_vs_oracle(pn, ora, b, k, a):
    x, t = _case(b, k, b * 31 + k)
    rc, want_l = ora.ls_ce_forward(x, t, a)
    assert rc == 0
    want_g = ora.ls_ce_backward(x, t, a)[1]
    bound = _bound(x, t, a)
    rc, gl, _ = _ls_gpu(pn, x, t, a, "fwd")
    assert rc == 0
    _loss_close(gl, want_l, bound)
    rc, _, gg = _ls_gpu(pn, x, t, a, "bwd")
    assert rc == 0
    rel_close(gg, want_g, 1e-12, 2e-15 / b, "ls_ce grad")
    rc, fl, fg = _ls_gpu(pn, x, t, a, "fused")
    assert rc == 0
    # the forward's exp comes from its LDS table (~3 ulp), the fused kernel's
    # from the library (it keeps every e for the gradient): the row sums can
    # differ in their last bits, so the losses agree to well inside the bar
    _loss_close(fl, gl, bound, tol=1e-13)
    # backward and fused share the exp, the sums and the gradient formula
    assert np.array_equal(fg.view(np.uint64), gg.view(np.uint64))
    if ora.ref() is not None:  # the reference's own C, when it travelled with the tree
        _loss_close(gl, ora.ls_ce_forward(x, t, a, use_ref=True)[1], bound)


def test_ls_ce_special_values(pn, ora):
    x, t = _case(6, 9, 5, special=True)
    for a in (0.0, 0.3, 1.0):
        want_l = ora.ls_ce_forward(x, t, a)[1]
        want_g = ora.ls_ce_backward(x, t, a)[1]
        rc, gl, gg = _ls_gpu(pn, x, t, a, "fused")
        assert rc == 0
        _loss_close(gl, want_l, _bound(x, t, a))
        rel_close(gg, want_g, 1e-12, 2e-15 / 6, "ls_ce grad special")


def test_ls_ce_errors(pn):
    lib = pn.core._lib
    x = np.zeros((2, 3))
    loss = ctypes.c_double()
    for t, a in [(np.array([0, 3]), 0.1), (np.array([-1, 0]), 0.1), (np.array([0, 1]), -0.1),
                 (np.array([0, 1]), 1.5), (np.array([0, 1]), float("nan"))]:
        t = t.astype(np.int64)
        assert lib.label_smoothing_ce_forward(x.ctypes.data, t.ctypes.data, 2, 3, a, ctypes.byref(loss)) == -1
    t = np.array([0, 1], dtype=np.int64)
    assert lib.label_smoothing_ce_forward(None, t.ctypes.data, 2, 3, 0.1, ctypes.byref(loss)) == -1
    assert lib.label_smoothing_ce_forward(x.ctypes.data, t.ctypes.data, 0, 3, 0.1, ctypes.byref(loss)) == -1
    assert lib.label_smoothing_ce_backward(x.ctypes.data, t.ctypes.data, 2, 3, 0.1, None) == -1
    # still usable after an error
    assert lib.label_smoothing_ce_forward(x.ctypes.data, t.ctypes.data, 2, 3, 0.1, ctypes.byref(loss)) == 0
    assert abs(loss.value - math.log(3.0)) < 1e-15


def test_ls_ce_device_pointers_and_f32(pn, ora):
    torch = pytest.importorskip("torch")
    b, k = 4096, 1000
    x, t = _case(b, k, 77)
    xt = torch.from_numpy(x).cuda()
    tt = torch.from_numpy(t).cuda()
    g = torch.empty_like(xt)
    loss = ctypes.c_double()
    torch.cuda.synchronize()
    lib = pn.core._lib
    assert lib.label_smoothing_ce_fused(xt.data_ptr(), tt.data_ptr(), b, k, 0.1, ctypes.byref(loss), g.data_ptr()) == 0
    pn.synchronize()
    want_l = ora.ls_ce_forward(x, t, 0.1)[1]
    want_g = ora.ls_ce_backward(x, t, 0.1)[1]
    _loss_close(loss.value, want_l, _bound(x, t, 0.1))
    rel_close(g.cpu().numpy(), want_g, 1e-12, 2e-15 / b, "device grad")
    # f32 logits: the reference formula on the exactly widened values, grad rounded to float
    x32 = x.astype(np.float32)
    x32t = torch.from_numpy(x32).cuda()
    g32 = torch.empty_like(x32t)
    torch.cuda.synchronize()
    assert lib.label_smoothing_ce_fused_f32(x32t.data_ptr(), tt.data_ptr(), b, k, 0.1, ctypes.byref(loss),
                                            g32.data_ptr()) == 0
    pn.synchronize()
    xw = x32.astype(np.float64)
    want_l = ora.ls_ce_forward(xw, t, 0.1)[1]
    want_g = ora.ls_ce_backward(xw, t, 0.1)[1].astype(np.float32)
    assert abs(loss.value - want_l) <= 2e-7 * _bound(xw, t, 0.1)
    rel_close(g32.cpu().numpy(), want_g, 1e-5, 2e-7 / b, "f32 grad")


@pytest.mark.parametrize("dt", [np.float32, np.float64])
@pytest.mark.parametrize("b,k", [(1, 2), (100, 10), (1000, 1000), (33, 5000)])
def test_cross_entropy_loss(pn, ora, dt, b, k):
    rng = np.random.default_rng(b + k)
    x = rng.normal(0, 3, (b, k)).astype(dt)
    tv = rng.integers(0, k, b).astype(dt)
    got = pn.CrossEntropyLoss()(pn.Tensor.from_numpy(x), pn.Tensor.from_numpy(tv))
    rc, want = ora.ce_loss(x, tv)
    assert rc == 0
    xd = x.astype(np.float64)
    m = xd.max(axis=1, keepdims=True)
    p = np.exp(xd - m) / np.exp(xd - m).sum(axis=1, keepdims=True)
    exact = float(np.mean(-np.log(p[np.arange(b), tv.astype(np.int64)] + 1e-7)))
    if dt == np.float64:
        assert abs(got - want) <= 1e-12 * abs(want)
    else:
        # p_target is a float: near 1 its rounding (6e-8) is absolute in the loss
        assert abs(got - exact) <= 2e-6 * abs(exact) + 2e-7
        assert abs(want - exact) <= 1e-3 * abs(exact) + 2e-7  # the reference's float order, reported


def test_cross_entropy_loss_errors(pn):
    lib = pn.core._lib
    x = pn.Tensor.from_numpy(np.zeros((4, 3), dtype=np.float32))
    loss = ctypes.c_double()
    bad = pn.Tensor.from_numpy(np.array([0, 1, 3, 0], dtype=np.float32))
    assert lib.neural_cross_entropy_loss(x._ptr, bad._ptr, ctypes.byref(loss)) == pn.NeuralError.INVALID_ARGUMENT
    nan = pn.Tensor.from_numpy(np.array([0, np.nan, 1, 0], dtype=np.float32))
    assert lib.neural_cross_entropy_loss(x._ptr, nan._ptr, ctypes.byref(loss)) == pn.NeuralError.INVALID_ARGUMENT
    f64 = pn.Tensor.from_numpy(np.zeros(4))
    assert lib.neural_cross_entropy_loss(x._ptr, f64._ptr, ctypes.byref(loss)) == pn.NeuralError.DTYPE_MISMATCH
    short = pn.Tensor.from_numpy(np.zeros(3, dtype=np.float32))
    assert lib.neural_cross_entropy_loss(x._ptr, short._ptr, ctypes.byref(loss)) == pn.NeuralError.SHAPE_MISMATCH
    assert lib.neural_cross_entropy_loss(None, short._ptr, ctypes.byref(loss)) == pn.NeuralError.NULL_POINTER
    ok = pn.Tensor.from_numpy(np.array([0, 1.9, 2, 0], dtype=np.float32))  # 1.9 truncates to class 1
    assert lib.neural_cross_entropy_loss(x._ptr, ok._ptr, ctypes.byref(loss)) == 0
    assert abs(loss.value - (-math.log(1.0 / 3.0 + 1e-7))) < 1e-6


def test_label_smoothing_module(pn, ora):
    m = pn.LabelSmoothingCrossEntropy(num_classes=4, smoothing=0.2)
    logits = [0.5, -1.0, 2.0, 0.0, 1.0, 1.0, -2.0, 3.0]
    got = m(logits, [2, 3])
    want = ora.ls_ce_forward(np.array(logits).reshape(2, 4), np.array([2, 3]), 0.2)[1]
    assert abs(got - want) <= 1e-14 * abs(want)
    g = (ctypes.c_double * 8)()
    m.backward_f64(ctypes.cast(g, ctypes.c_void_p))
    rel_close(np.frombuffer(g, dtype=np.float64).reshape(2, 4),
              ora.ls_ce_backward(np.array(logits).reshape(2, 4), np.array([2, 3]), 0.2)[1], 1e-12, 1e-15, "module")


def test_label_smoothing_module_device_loss(pn):
    """The module's _dev methods: the host forms' loss and gradient, the loss
    read from device memory after one synchronisation; a host pointer raises."""
    torch = pytest.importorskip("torch")
    m = pn.LabelSmoothingCrossEntropy(num_classes=37, smoothing=0.15)
    x, t = _case(300, 37, 5)
    xt, tt = torch.from_numpy(x).cuda(), torch.from_numpy(t).cuda()
    g1, g2 = torch.empty_like(xt), torch.empty_like(xt)
    loss = torch.zeros(2, dtype=torch.float64, device="cuda")
    torch.cuda.synchronize()
    want = m.forward_backward_f64(xt.data_ptr(), tt.data_ptr(), 300, g1.data_ptr())
    m.forward_f64_dev(xt.data_ptr(), tt.data_ptr(), 300, loss.data_ptr())
    m.forward_backward_f64_dev(xt.data_ptr(), tt.data_ptr(), 300, g2.data_ptr(), loss.data_ptr() + 8)
    pn.synchronize()
    assert loss.cpu().tolist() == [want, want]
    assert torch.equal(g1, g2)
    with pytest.raises(pn.NeuralException):
        m.forward_f64_dev(x.ctypes.data, tt.data_ptr(), 300, loss.data_ptr())


@pytest.mark.parametrize("k", [1000, 1024])
def test_ls_ce_loss_left_in_device_memory(pn, k):
    """The _dev forms (no reference counterpart): the host-returning forms'
    loss and gradient bits, the loss stored in device memory; three calls
    queue without waiting; a target out of range gives a NaN loss and does
    not reach the next host-returning call; argument errors return -1."""
    torch = pytest.importorskip("torch")
    lib = pn.core._lib
    b = 4096
    x, t = _case(b, k, 91)  # finite logits: a NaN loss below can only come from the bad target
    xt, tt = torch.from_numpy(x).cuda(), torch.from_numpy(t).cuda()
    x32t = xt.float()
    g_host, g_dev = torch.empty_like(xt), torch.full_like(xt, 7.0)
    g32_host, g32_dev = torch.empty_like(x32t), torch.full_like(x32t, 7.0)
    losses = torch.full((4,), 7.0, dtype=torch.float64, device="cuda")
    torch.cuda.synchronize()
    want = [ctypes.c_double() for _ in range(3)]
    assert lib.label_smoothing_ce_forward(xt.data_ptr(), tt.data_ptr(), b, k, 0.1, ctypes.byref(want[0])) == 0
    assert lib.label_smoothing_ce_fused(xt.data_ptr(), tt.data_ptr(), b, k, 0.1, ctypes.byref(want[1]),
                                        g_host.data_ptr()) == 0
    assert lib.label_smoothing_ce_fused_f32(x32t.data_ptr(), tt.data_ptr(), b, k, 0.1, ctypes.byref(want[2]),
                                            g32_host.data_ptr()) == 0
    pn.synchronize()
    assert all(math.isfinite(w.value) for w in want)
    p = losses.data_ptr()
    assert lib.label_smoothing_ce_forward_dev(xt.data_ptr(), tt.data_ptr(), b, k, 0.1, p) == 0
    assert lib.label_smoothing_ce_fused_dev(xt.data_ptr(), tt.data_ptr(), b, k, 0.1, p + 8, g_dev.data_ptr()) == 0
    assert lib.label_smoothing_ce_fused_f32_dev(x32t.data_ptr(), tt.data_ptr(), b, k, 0.1, p + 16,
                                                g32_dev.data_ptr()) == 0
    pn.synchronize()
    got = losses.cpu().numpy()
    same_bits(got[:3], np.array([w.value for w in want]))
    assert got[3] == 7.0  # nothing written past the three losses
    same_bits(g_dev.cpu().numpy(), g_host.cpu().numpy())
    same_bits(g32_dev.cpu().numpy(), g32_host.cpu().numpy())
    # a target out of range: a NaN loss, and the next host-returning call is clean
    t2 = t.copy()
    t2[17] = k
    tt2 = torch.from_numpy(t2).cuda()
    torch.cuda.synchronize()
    assert lib.label_smoothing_ce_forward_dev(xt.data_ptr(), tt2.data_ptr(), b, k, 0.1, p) == 0
    pn.synchronize()
    assert math.isnan(losses[0].item())
    again = ctypes.c_double()
    assert lib.label_smoothing_ce_forward(xt.data_ptr(), tt.data_ptr(), b, k, 0.1, ctypes.byref(again)) == 0
    same_bits(np.array(again.value), np.array(want[0].value))
    # argument errors: host memory, misalignment, NULL, sizes, smoothing
    assert lib.label_smoothing_ce_forward_dev(x.ctypes.data, tt.data_ptr(), b, k, 0.1, p) == -1
    assert lib.label_smoothing_ce_forward_dev(xt.data_ptr(), t.ctypes.data, b, k, 0.1, p) == -1
    host_loss = np.zeros(1)
    assert lib.label_smoothing_ce_forward_dev(xt.data_ptr(), tt.data_ptr(), b, k, 0.1, host_loss.ctypes.data) == -1
    assert lib.label_smoothing_ce_forward_dev(xt.data_ptr(), tt.data_ptr(), b, k, 0.1, p + 4) == -1
    assert lib.label_smoothing_ce_forward_dev(xt.data_ptr(), tt.data_ptr(), b, k, 0.1, None) == -1
    assert lib.label_smoothing_ce_fused_dev(xt.data_ptr(), tt.data_ptr(), b, k, 0.1, p, None) == -1
    assert lib.label_smoothing_ce_forward_dev(xt.data_ptr(), tt.data_ptr(), 0, k, 0.1, p) == -1
    assert lib.label_smoothing_ce_forward_dev(xt.data_ptr(), tt.data_ptr(), b, k, 1.5, p) == -1
    pn.synchronize()
    assert math.isnan(losses[0].item()) and losses[3].item() == 7.0  # untouched by the refused calls


# Class counts at the edges of the row kernels (4 or 16 lanes per row up to 259
# f32 values; 2 .. 16 vectors per lane in a wave, 8 / 16 in a block of 256, 16
# and 16 + 9 (the 9 in LDS) in 512, 24 in 1024, two reads beyond); f64 at half.
_EDGES = [1, 2, 3, 15, 16, 19, 20, 64, 67, 68, 256, 259, 260, 511, 513, 1023, 1025, 2049, 4096, 4099, 4101, 8193, 16385,
          32768, 32785, 49153, 51200, 51217, 98304, 98321, 120001]


@pytest.mark.parametrize("k", _EDGES)
@pytest.mark.parametrize("dt", ["float32", "float64"])
def test_row_kernel_edges(pn, dt, k):
    """Fused, backward and forward smoothed CE and the tensor CE at each row
    kernel's edges against the float64 formula, at several element offsets of
    logits and gradient, the target in the first, last and inner values, -inf
    logits, a NaN row and a row of only -inf.  Bounds: those of the module."""
    import torch
    lib = pn.core._lib
    T = getattr(torch, dt)
    k = k if dt == "float32" else max(1, (k + 1) // 2)
    b = 9
    rng = np.random.default_rng(k)
    x = rng.normal(0, 3, (b, k)).astype(dt)
    t = rng.integers(0, k, b)
    t[:4] = [0, k - 1, max(0, k - 2), min(k - 1, 17)]
    if k > 4:
        x[5, : k // 2] = -np.inf
        t[5] = k - 1
    special = [5, 6, 7]  # the loss of these rows is not finite
    x[6, k // 2] = np.nan
    x[7] = -np.inf
    fine = [r for r in range(b) if r not in special]
    x64, a = x.astype(np.float64), 0.1
    f64 = dt == "float64"
    pn.set_stream(torch.cuda.current_stream().cuda_stream)
    try:
        for rows, oi, og in ((fine, 0, 0), (fine, 1, 3), (fine, 3, 0), (list(range(b)), 1, 1)):
            n = len(rows)
            bx, bg = (torch.full((n * k + 8,), 7.0, dtype=T, device="cuda") for _ in range(2))
            X, G = bx[oi:oi + n * k].view(n, k), bg[og:og + n * k].view(n, k)
            X.copy_(torch.from_numpy(x[rows]))
            tt = torch.from_numpy(t[rows]).cuda()
            loss = torch.zeros((), dtype=torch.float64, device="cuda")
            args = (X.data_ptr(), tt.data_ptr(), n, k, a)
            fn = lib.label_smoothing_ce_fused_dev if f64 else lib.label_smoothing_ce_fused_f32_dev
            assert fn(*args, loss.data_ptr(), G.data_ptr()) == 0
            xr = x64[rows]
            with np.errstate(all="ignore"):
                d = xr - np.max(np.where(np.isnan(xr), -np.inf, xr), axis=1, keepdims=True)
                e = np.exp(d)
                s = e.sum(axis=1, keepdims=True)
                st = np.full((n, k), a / k)
                st[np.arange(n), t[rows]] += 1 - a
                want = (e / s - st) / n
                want_loss = -(st * (d - np.log(s))).sum() / n
            got = G.cpu().numpy().astype(np.float64)
            assert np.array_equal(np.isnan(got), np.isnan(want))
            ok = ~np.isnan(want)
            bound = 1e-12 * np.abs(want[ok]) + 2e-15 / n if f64 else 1e-5 * np.abs(want[ok]) + 2e-7 / n
            assert np.all(np.abs(got[ok] - want[ok]) <= bound), (oi, og)
            if np.isfinite(want_loss):
                scale = _bound(xr, t[rows], a)
                assert abs(loss.item() - want_loss) <= (1e-12 if f64 else 2e-6) * scale
            else:
                assert not np.isfinite(loss.item())
            edge = torch.cat([bg[:og], bg[og + n * k:]])
            assert bool((edge == 7.0).all())  # nothing written outside the rows
            if f64:
                fused = G.clone()
                G.fill_(0.0)
                assert lib.label_smoothing_ce_backward(*args, G.data_ptr()) == 0
                assert torch.equal(fused.view(torch.int64), G.view(torch.int64))
                fwd = torch.zeros((), dtype=torch.float64, device="cuda")
                assert lib.label_smoothing_ce_forward_dev(*args, fwd.data_ptr()) == 0
                if np.isfinite(want_loss):
                    assert abs(fwd.item() - want_loss) <= 1e-12 * scale
            if rows is fine:
                got_ce = ctypes.c_double()
                tx, tv = pn.Tensor.from_torch(X), pn.Tensor.from_torch(tt.to(T))
                assert lib.neural_cross_entropy_loss(tx._ptr, tv._ptr, ctypes.byref(got_ce)) == 0
                want_ce = np.mean(-np.log((e / s)[np.arange(n), t[rows]] + 1e-7))
                assert abs(got_ce.value - want_ce) <= (1e-12 * abs(want_ce) + 1e-15 if f64
                                                       else 2e-6 * abs(want_ce) + 2e-7)
        # a target outside [0, k): NaN loss, the other rows' gradients written
        tt[1] = k
        G.fill_(7.0)
        assert fn(*args, loss.data_ptr(), G.data_ptr()) == 0
        assert np.isnan(loss.item()) and bool((G[1] == 7.0).all()) and not bool((G[0] == 7.0).any())
    finally:
        pn.set_stream(None)


@pytest.mark.parametrize("k", [257, 513, 1001, 4099, 8193, 33001, 98311])
@pytest.mark.parametrize("dt", ["float64", "float32"])
def test_bits_do_not_depend_on_the_address(pn, dt, k):
    """Loss and gradient bits of the _dev form, whatever element the gradient
    starts at, equal the host-returning form's (whose gradient is staged in a
    block of its own) and, in f64, the backward's; equal rows have equal
    gradients, though rows of an odd width start at different addresses."""
    import torch
    lib = pn.core._lib
    T = getattr(torch, dt)
    n, a, f64 = 5, 0.1, dt == "float64"
    rng = np.random.default_rng(k)
    x = np.repeat(rng.normal(0, 3, (1, k)), n, axis=0).astype(dt)
    t = np.full(n, k // 3, dtype=np.int64)
    bits = np.int64 if f64 else np.int32
    host_g, host_loss = np.empty((n, k), dtype=dt), ctypes.c_double()
    fused = lib.label_smoothing_ce_fused if f64 else lib.label_smoothing_ce_fused_f32
    assert fused(x.ctypes.data, t.ctypes.data, n, k, a, ctypes.byref(host_loss), host_g.ctypes.data) == 0
    for r in range(1, n):
        assert np.array_equal(host_g[0].view(bits), host_g[r].view(bits))
    dev = lib.label_smoothing_ce_fused_dev if f64 else lib.label_smoothing_ce_fused_f32_dev
    pn.set_stream(torch.cuda.current_stream().cuda_stream)
    try:
        tt = torch.from_numpy(t).cuda()
        loss = torch.zeros((), dtype=torch.float64, device="cuda")
        for oi, og in ((0, 0), (0, 1), (1, 3), (3, 0), (2, 7)):
            bx, bg = (torch.zeros(n * k + 8, dtype=T, device="cuda") for _ in range(2))
            X, G = bx[oi:oi + n * k], bg[og:og + n * k]
            X.copy_(torch.from_numpy(x).flatten())
            assert dev(X.data_ptr(), tt.data_ptr(), n, k, a, loss.data_ptr(), G.data_ptr()) == 0
            assert np.array_equal(G.cpu().numpy().view(bits), host_g.ravel().view(bits)), (oi, og)
            assert loss.item() == host_loss.value
            if f64:
                G.zero_()
                assert lib.label_smoothing_ce_backward(X.data_ptr(), tt.data_ptr(), n, k, a, G.data_ptr()) == 0
                assert np.array_equal(G.cpu().numpy().view(bits), host_g.ravel().view(bits)), (oi, og)
    finally:
        pn.set_stream(None)


@pytest.mark.parametrize("k", [4097, 4098, 4099, 4100, 8193])
def test_wide_f32_rows_round_once(pn, k):
    """Rows of more than 4096 f32 classes form the gradient in double and round
    once.  Equal logits make every e exactly 1 and the sum exactly k, so only
    that forming is left: (1/n) (1/k - st) in double, rounded to float, where
    float arithmetic loses the digits that cancel (smoothing 0.9)."""
    import torch
    lib = pn.core._lib
    n, a = 3, 0.9
    x = torch.full((n, k), 1.25, dtype=torch.float32, device="cuda")
    g, loss = torch.zeros_like(x), torch.zeros((), dtype=torch.float64, device="cuda")
    t = torch.tensor([0, k // 2, k - 1], device="cuda")
    torch.cuda.synchronize()
    assert lib.label_smoothing_ce_fused_f32_dev(x.data_ptr(), t.data_ptr(), n, k, a, loss.data_ptr(), g.data_ptr()) == 0
    pn.synchronize()
    st = np.full((n, k), a / k)
    st[np.arange(n), t.cpu().numpy()] += 1.0 - a
    want = ((1.0 / n) * (1.0 / k - st)).astype(np.float32)
    got = g.cpu().numpy()
    # double forming: 2^-24 of the value and what double rounding leaves of the cancelled terms
    assert np.all(np.abs(got.astype(np.float64) - want) <= 2.0 ** -23 * np.abs(want))


@pytest.mark.parametrize("k", [2049, 2050, 2051])
def test_wide_f64_forward_exp(pn, k):
    """Past 2048 f64 classes the forward takes the library's exp, as the fused
    form does, and not the table's (about 3 ulp): the same loss bits.  One row
    a call, two classes that count (loss = log(1 + e^y)), so that a last bit of
    e^y shows."""
    import torch
    lib = pn.core._lib
    tt = torch.zeros(1, dtype=torch.int64, device="cuda")
    xt = torch.full((1, k), -800.0, dtype=torch.float64, device="cuda")
    g = torch.empty_like(xt)
    fwd, fused = ctypes.c_double(), ctypes.c_double()
    for y in np.linspace(-1.0, -0.01, 100):
        xt[0, 0], xt[0, k // 2] = 0.0, y
        torch.cuda.synchronize()
        assert lib.label_smoothing_ce_forward(xt.data_ptr(), tt.data_ptr(), 1, k, 0.0, ctypes.byref(fwd)) == 0
        assert lib.label_smoothing_ce_fused(xt.data_ptr(), tt.data_ptr(), 1, k, 0.0, ctypes.byref(fused),
                                            g.data_ptr()) == 0
        assert fwd.value == fused.value, y


@pytest.mark.parametrize("b", [2048, 2049, 4096, 4097, 8191, 32768, 32769])
def test_loss_sum_over_batches(pn, b):
    """The mean over the rows' losses at the batch sizes where the summing pass
    changes form (a wave, a block, segments); the _dev form gives the same
    bits.  Bounds: those of the module."""
    import torch
    lib = pn.core._lib
    k, a = 5, 0.1
    x, t = _case(b, k, b)
    xt, tt = torch.from_numpy(x).cuda(), torch.from_numpy(t).cuda()
    g, dev = torch.empty_like(xt), torch.zeros(2, dtype=torch.float64, device="cuda")
    torch.cuda.synchronize()
    fwd, fused, ce = (ctypes.c_double() for _ in range(3))
    args = (xt.data_ptr(), tt.data_ptr(), b, k, a)
    assert lib.label_smoothing_ce_forward(*args, ctypes.byref(fwd)) == 0
    assert lib.label_smoothing_ce_fused(*args, ctypes.byref(fused), g.data_ptr()) == 0
    assert lib.label_smoothing_ce_forward_dev(*args, dev.data_ptr()) == 0
    assert lib.label_smoothing_ce_fused_dev(*args, dev.data_ptr() + 8, g.data_ptr()) == 0
    pn.synchronize()
    same_bits(dev.cpu().numpy(), np.array([fwd.value, fused.value]))
    lsm = x - x.max(axis=1, keepdims=True)
    lsm -= np.log(np.exp(lsm).sum(axis=1, keepdims=True))
    st = np.full((b, k), a / k)
    st[np.arange(b), t] += 1 - a
    want = -(st * lsm).sum() / b
    for got in (fwd.value, fused.value):
        assert abs(got - want) <= 1e-12 * _bound(x, t, a)
    for dt, rel, floor in ((np.float64, 1e-12, 0.0), (np.float32, 2e-6, 2e-7)):
        tx, tv = pn.Tensor.from_numpy(x.astype(dt)), pn.Tensor.from_numpy(t.astype(dt))
        assert lib.neural_cross_entropy_loss(tx._ptr, tv._ptr, ctypes.byref(ce)) == 0
        x64 = x.astype(dt).astype(np.float64)
        p = np.exp(x64 - x64.max(axis=1, keepdims=True))
        want_ce = np.mean(-np.log((p / p.sum(axis=1, keepdims=True))[np.arange(b), t] + 1e-7))
        assert abs(ce.value - want_ce) <= rel * abs(want_ce) + floor


@pytest.mark.parametrize("k", [10, 64, 513, 1001, 2048, 4099, 8193, 33001, 49152, 98311])
@pytest.mark.parametrize("dt", ["float64", "float32"])
def test_fused_in_place(pn, dt, k):
    """The gradient written over the logits: same loss and gradient bits."""
    import torch
    lib = pn.core._lib
    n, f64 = 9, dt == "float64"
    fn = lib.label_smoothing_ce_fused_dev if f64 else lib.label_smoothing_ce_fused_f32_dev
    rng = np.random.default_rng(k)
    x = torch.from_numpy(rng.normal(0, 3, (n, k)).astype(dt)).cuda()
    t = torch.from_numpy(rng.integers(0, k, n)).cuda()
    g, loss = torch.empty_like(x), torch.zeros(2, dtype=torch.float64, device="cuda")
    torch.cuda.synchronize()
    assert fn(x.data_ptr(), t.data_ptr(), n, k, 0.1, loss.data_ptr(), g.data_ptr()) == 0
    assert fn(x.data_ptr(), t.data_ptr(), n, k, 0.1, loss.data_ptr() + 8, x.data_ptr()) == 0
    pn.synchronize()
    assert loss[0].item() == loss[1].item()
    same_bits(x.cpu().numpy(), g.cpu().numpy())

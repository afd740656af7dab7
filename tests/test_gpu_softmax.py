"""Row softmax / log-softmax parity.

Contract: REL32 (|g - r| <= 1e-5 |r|) for f32 outputs and REL64
(|g - r| <= 1e-12 |r| + 1e-15) for f64, where r is the fp64-exact softmax
(numpy, float64 math).  The oracle's sequential-order restatement of
node_softmax / metrics_losses.c:47-64 is held to the same bound.  A NaN in a
row makes the whole row NaN, as in the reference.
"""

import numpy as np
import pytest

from conftest import GPU, rel_close

pytestmark = GPU


def _exact(x, log):
    x64 = x.astype(np.float64)
    m = np.max(np.where(np.isnan(x64), -np.inf, x64), axis=1, keepdims=True)
    e = np.exp(x64 - m)
    s = np.sum(e, axis=1, keepdims=True)
    return (x64 - m) - np.log(s) if log else e / s


def _run(pn, x, log):
    mod = pn.LogSoftmax() if log else pn.Softmax()
    return mod(pn.Tensor.from_numpy(x)).numpy()


@pytest.mark.parametrize("rows,cols", [(65536, 1024), (100, 1000), (33, 4096), (7, 5000), (9, 3), (1, 1)])
@pytest.mark.parametrize("log", [False, True])
def test_softmax_f32(pn, ora, rows, cols, log):
    rng = np.random.default_rng(rows + cols + int(log))
    x = rng.normal(0, 3, (rows, cols)).astype(np.float32)
    got = _run(pn, x, log)
    want = _exact(x, log)
    rel_close(got, want, 1e-5, 0.0, "gpu vs fp64 exact")
    if rows * cols <= 1 << 22:
        rel_close(ora.softmax_rows(x, log), want, 1e-5, 0.0, "oracle vs fp64 exact")


@pytest.mark.parametrize("rows,cols", [(4096, 1024), (50, 2048), (5, 3001)])
@pytest.mark.parametrize("log", [False, True])
def test_softmax_f64(pn, ora, rows, cols, log):
    rng = np.random.default_rng(cols)
    x = rng.normal(0, 3, (rows, cols))
    got = _run(pn, x, log)
    rel_close(got, _exact(x, log), 1e-12, 1e-15, "gpu vs fp64 exact")
    rel_close(got, ora.softmax_rows(x, log), 1e-12, 1e-15, "gpu vs oracle")


def test_softmax_special_rows(pn, ora):
    x = np.random.default_rng(5).normal(0, 3, (6, 256)).astype(np.float32)
    x[1, 17] = np.nan
    x[2, :] = -np.inf
    x[3, 5] = np.inf
    x[4, :] = 30.0
    x[5, 0] = 80.0
    for log in (False, True):
        got = _run(pn, x, log)
        want = ora.softmax_rows(x, log)
        assert np.array_equal(np.isnan(got), np.isnan(want))
        ok = ~np.isnan(want)
        rel_close(got[ok], want[ok], 1e-5, 1e-30, "special rows")
        assert np.all(np.isnan(got[1])) and np.all(np.isnan(got[2]))


def test_softmax_errors(pn):
    a = pn.Tensor.create([4, 8])
    b = pn.Tensor.create([4, 8], pn.float64)
    assert pn.core._lib.neural_softmax(b._ptr, a._ptr) == pn.NeuralError.DTYPE_MISMATCH
    c = pn.Tensor.create([5, 8])
    assert pn.core._lib.neural_softmax(c._ptr, a._ptr) == pn.NeuralError.SHAPE_MISMATCH


# Widths at the edges of the row kernels (4 or 16 lanes per row up to 256
# values; vectors held per lane: 2 .. 16 in a wave, 8 / 16 / 25 in blocks of 256 / 512, 16 / 24 in 1024, two reads beyond),
# for f32; the f64 edges lie at half of each.
_EDGES = [1, 2, 3, 5, 15, 16, 19, 20, 63, 64, 67, 68, 127, 129, 255, 256, 257, 511, 513, 1023, 1025, 2047, 2049, 4093, 4096, 4099, 8191, 8197, 16383, 16385,
          32767, 32769, 51197, 51201, 65535, 65537, 98301, 98304, 98305, 98311, 140003]


@pytest.mark.parametrize("cols", _EDGES)
@pytest.mark.parametrize("dt", ["float32", "float64"])
def test_row_kernel_edges(pn, dt, cols):
    """Softmax and log-softmax at each kernel's edges, rows starting at any
    element offset, against the float64 formula (REL32 / REL64); -inf entries,
    a NaN row and an all -inf row among them, and in place."""
    import torch
    T = getattr(torch, dt)
    cols = cols if dt == "float32" else max(1, (cols + 1) // 2)
    rows = 7 if cols > 1024 else 71
    g = torch.Generator().manual_seed(cols)
    x = (torch.randn((rows, cols), generator=g, dtype=torch.float64) * 3).to(T)
    x[1, : cols // 2] = -float("inf")
    x[3, cols - 1] = float("nan")
    x[4] = -float("inf")
    x[5, cols - 1] = 40.0  # the maximum in the last (scalar) value
    x64 = x.double()
    e = torch.exp(x64 - x64.max(1, keepdim=True)[0])
    s = e.sum(1, keepdim=True)
    rel, floor = (1e-5, 1e-6) if dt == "float32" else (1e-12, 1e-15)
    pn.set_stream(torch.cuda.current_stream().cuda_stream)
    try:
        for off_in, off_out, log in ((0, 0, False), (1, 0, True), (0, 3, False), (1, 1, True), (None, None, False)):
            buf = torch.zeros(rows * cols + 8, dtype=T, device="cuda")
            out = torch.full((rows * cols + 8,), 7.0, dtype=T, device="cuda")
            if off_in is None:  # in place
                off_in = off_out = 1
                out = buf
                buf[0] = buf[1 + rows * cols:] = 7.0
            xi, yo = (b[o:o + rows * cols].view(rows, cols) for b, o in ((buf, off_in), (out, off_out)))
            xi.copy_(x)
            tx, ty = pn.Tensor.from_torch(xi), pn.Tensor.from_torch(yo)
            f = pn.core._lib.neural_log_softmax if log else pn.core._lib.neural_softmax
            assert f(ty._ptr, tx._ptr) == 0
            got = yo.cpu().double()
            want = (x64 - x64.max(1, keepdim=True)[0]) - torch.log(s) if log else e / s
            assert torch.equal(torch.isnan(got), torch.isnan(want)) and torch.equal(torch.isinf(got), torch.isinf(want))
            fin = torch.isfinite(want)
            bound = rel * want[fin].abs() + (floor if log or dt == "float64" else 0.0)
            assert bool(((got[fin] - want[fin]).abs() <= bound).all()), (off_in, off_out, log)
            edge = torch.cat([out[:off_out], out[off_out + rows * cols:]])
            assert bool((edge == 7.0).all())  # nothing written outside the rows
    finally:
        pn.set_stream(None)


def test_timed_launch(pn):
    """neural_hip_time_next_launch: the events ride on the chosen launch of the
    calling thread (elapsed time > 0, outputs unchanged), are used once, can
    skip launches (the combine launch of a whole-tensor sum is skip = 1) and
    be cancelled; null events and negative skips are rejected."""
    import ctypes
    from pathlib import Path
    import torch
    hip = ctypes.CDLL(str(Path(torch.__file__).parent / "lib" / "libamdhip64.so"))
    hip.hipEventCreate.argtypes = [ctypes.POINTER(ctypes.c_void_p)]
    hip.hipEventElapsedTime.argtypes = [ctypes.POINTER(ctypes.c_float), ctypes.c_void_p, ctypes.c_void_p]
    hip.hipEventDestroy.argtypes = [ctypes.c_void_p]
    lib = pn.core._lib
    rng = np.random.default_rng(41)
    x = rng.normal(0, 3, (512, 1024)).astype(np.float32)
    tx = pn.Tensor.from_numpy(x)
    y_plain = pn.Tensor.create(tx.shape, tx.dtype)
    assert lib.neural_softmax(y_plain._ptr, tx._ptr) == 0
    s = torch.cuda.current_stream()
    lib.neural_hip_set_stream(ctypes.c_void_p(s.cuda_stream))
    ev = []
    try:
        def pair():
            e0, e1 = ctypes.c_void_p(), ctypes.c_void_p()
            assert hip.hipEventCreate(ctypes.byref(e0)) == 0 and hip.hipEventCreate(ctypes.byref(e1)) == 0
            ev.extend([e0, e1])
            return e0, e1

        def elapsed(e0, e1):
            ms = ctypes.c_float()
            assert hip.hipEventElapsedTime(ctypes.byref(ms), e0, e1) == 0
            return ms.value

        e0, e1 = pair()
        assert lib.neural_hip_time_next_launch(e0, e1, 0) == 0
        y = pn.Tensor.create(tx.shape, tx.dtype)
        assert lib.neural_softmax(y._ptr, tx._ptr) == 0
        torch.cuda.synchronize()
        assert elapsed(e0, e1) > 0.0
        assert np.array_equal(y.numpy(), y_plain.numpy())
        assert lib.neural_softmax(y._ptr, tx._ptr) == 0  # nothing armed: a plain launch
        assert np.array_equal(y.numpy(), y_plain.numpy())
        # a whole-tensor sum of 2^24 values is a segment launch and a combine launch
        big = pn.Tensor.from_numpy(rng.uniform(-1, 1, 1 << 24).astype(np.float32))
        r0 = ctypes.c_double()
        assert lib.neural_sum(big._ptr, ctypes.byref(r0)) == 0
        a0, a1 = pair()
        b0, b1 = pair()
        assert lib.neural_hip_time_next_launch(a0, a1, 0) == 0
        r1 = ctypes.c_double()
        assert lib.neural_sum(big._ptr, ctypes.byref(r1)) == 0
        assert lib.neural_hip_time_next_launch(b0, b1, 1) == 0
        r2 = ctypes.c_double()
        assert lib.neural_sum(big._ptr, ctypes.byref(r2)) == 0
        torch.cuda.synchronize()
        seg_ms, comb_ms = elapsed(a0, a1), elapsed(b0, b1)
        assert seg_ms > 0.0 and comb_ms > 0.0 and comb_ms < seg_ms, (seg_ms, comb_ms)
        assert r0.value == r1.value == r2.value
        # cancel: armed events are dropped unused
        c0, c1 = pair()
        assert lib.neural_hip_time_next_launch(c0, c1, 0) == 0
        assert lib.neural_hip_time_cancel() == 0
        assert lib.neural_softmax(y._ptr, tx._ptr) == 0
        torch.cuda.synchronize()
        ms = ctypes.c_float()
        assert hip.hipEventElapsedTime(ctypes.byref(ms), c0, c1) != 0  # never recorded
        hip.hipGetLastError()  # clear that error so the next library call does not report it
        assert lib.neural_hip_time_next_launch(None, e1, 0) == pn.NeuralError.NULL_POINTER
        assert lib.neural_hip_time_next_launch(e0, e1, -1) == pn.NeuralError.INVALID_ARGUMENT
    finally:
        lib.neural_hip_time_cancel()
        lib.neural_hip_reset_stream()
        for e in ev:
            hip.hipEventDestroy(e)


@pytest.mark.parametrize("cols", [577, 4099, 8191, 33001, 51203, 98301, 98311])
@pytest.mark.parametrize("dt", ["float32", "float64"])
def test_bits_do_not_depend_on_the_address(pn, dt, cols):
    """Equal rows have equal outputs, wherever the input and output start."""
    import torch
    T = getattr(torch, dt)
    cols = cols if dt == "float32" else (cols + 1) // 2 | 1
    g = torch.Generator().manual_seed(cols)
    row = (torch.randn((1, cols), generator=g, dtype=torch.float64) * 3).to(T).cuda()
    bits = torch.int32 if dt == "float32" else torch.int64
    pn.set_stream(torch.cuda.current_stream().cuda_stream)
    try:
        for f in (pn.core._lib.neural_softmax, pn.core._lib.neural_log_softmax):
            first = None
            for oi, oo in ((0, 0), (1, 3), (3, 2)):
                x, y = (torch.zeros(5 * cols + 8, dtype=T, device="cuda") for _ in range(2))
                X, Y = x[oi:oi + 5 * cols].view(5, cols), y[oo:oo + 5 * cols].view(5, cols)
                X.copy_(row.expand(5, cols))
                assert f(pn.Tensor.from_torch(Y)._ptr, pn.Tensor.from_torch(X)._ptr) == 0
                first = Y[0].clone() if first is None else first
                assert torch.equal(Y.contiguous().view(bits), first.view(bits).expand(5, cols)), (oi, oo)
    finally:
        pn.set_stream(None)

"""The F32 GEMM's tiles and rings against FP64: 32- and 64-row tiles, K of one
step to more than the LDS ring holds, split and unsplit, ragged rows and
features, a row past the FP32 limit.  |err| <= (cols + 2) 2^-24 sum |x||w|: one
rounding per addition of the longest chain."""
import ctypes as C

import numpy as np
import pytest

import oracle
import sr_go_tranformer_amd as srq

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ex():
    e = srq.Executor(0)
    yield e
    e.close()


@pytest.mark.parametrize("rows,cols,ns", [
    (3, 32, (17, 33)),               # one step, fewer features than a tile
    (130, 64, (32, 65, 300)),        # two steps
    (129, 160, (31, 64)),            # a slice of as many steps as the small ring and more
    (1000, 608, (17, 97)),           # split K, a shorter last slice
    (33000, 224, (17, 40, 66)),      # not split: y written directly, 64-row tiles
    (3072, 576, (129, 257)),
])
def test_f32_gemm(ex, rows, cols, ns):
    rng = oracle.RNG(rows + cols)
    dense = np.resize(rng.fill_normal(1 << 16, 0.02), rows * cols).reshape(rows, cols)
    w = srq.Weight.create(ex, dense, srq.F32)
    first = None
    for n in ns:
        x = np.resize(rng.fill_normal(1 << 15, 1.0), n * cols).reshape(n, cols).copy()
        x[:17] = np.resize(oracle.RNG(cols).fill_normal(4096, 1.0), 17 * cols).reshape(17, cols)
        x[n - 1, cols // 2] = 3e34
        print("f32 gemm", rows, cols, n, flush=True)
        got = srq.linear(ex, w, x)
        xd, wd = x.astype(np.float64), dense.astype(np.float64)
        want, bound = xd @ wd.T, (cols + 2) * 2.0 ** -24 * (np.abs(xd) @ np.abs(wd).T)
        assert (np.abs(got - want) <= bound).all(), n
        if first is None:
            first = got[:16]
        assert np.array_equal(got[:16].view(np.uint32), first.view(np.uint32)), n  # rows do not depend on n


def test_f32_gemm_unaligned_rows(ex):
    """Activations that start at any float, as a view into a larger buffer does:
    the bits of the aligned call (F32, Q8 and Q4)."""
    rng = oracle.RNG(3)
    rows, cols, n = 300, 512, 150
    dense = rng.fill_normal(rows * cols, 0.02).reshape(rows, cols)
    x = rng.fill_normal(n * cols, 1.0).reshape(n, cols)
    for fmt in (srq.F32, srq.Q8, srq.Q4):
        w = srq.Weight.create(ex, dense, fmt)
        for m in (1, 17, 32, n):
            print("unaligned", fmt, m, flush=True)
            want = srq.linear(ex, w, x[:m])
            xb = ex.upload(np.concatenate([np.zeros(1, np.float32), x[:m].ravel()]))
            yb = ex.empty(m * rows * 4)
            srq.check(srq.lib().srq_linear(ex.h, yb.ptr, C.c_void_p(xb.ptr.value + 4), w.h, m))
            got = yb.to_numpy(np.float32, (m, rows))
            assert np.array_equal(got.view(np.uint32), want.view(np.uint32)), (fmt, m)


@pytest.mark.parametrize("rows,cols,ns", [
    (3, 32, (17, 33)),           # one step: what follows it is loaded again, never used
    (130, 64, (32, 65, 300)),    # two steps
    (1000, 608, (17, 97)),       # split K, a shorter last slice
    (33000, 224, (40, 66)),      # not split, 64-row tiles
])
def test_f32_steps_through_registers(ex, rows, cols, ns):
    """F32 operands off a 16-byte boundary (activations, then also the values):
    the aligned call's bits, at the edges of the steps and tiles."""
    rng = oracle.RNG(rows + cols)
    dense = np.resize(rng.fill_normal(1 << 16, 0.02), rows * cols).reshape(rows, cols).astype(np.float32)
    w = srq.Weight.create(ex, dense, srq.F32)
    one = np.zeros(1, np.float32)
    vb = ex.upload(np.concatenate([one, dense.ravel()]))
    h = C.c_void_p()
    srq.check(srq.lib().srq_weight_wrap(srq.F32, rows, cols, C.c_void_p(vb.ptr.value + 4), None, C.byref(h)))
    wrapped = srq.Weight(h)
    for n in ns:
        print("f32 registers", rows, cols, n, flush=True)
        x = np.resize(rng.fill_normal(1 << 15, 1.0), n * cols).reshape(n, cols).copy()
        x[n - 1, cols // 2] = 3e34
        want = srq.linear(ex, w, x)
        xb = ex.upload(np.concatenate([one, x.ravel()]))
        for weights in (w, wrapped):
            yb = ex.empty(n * rows * 4)
            srq.check(srq.lib().srq_linear(ex.h, yb.ptr, C.c_void_p(xb.ptr.value + 4), weights.h, n))
            assert np.array_equal(yb.to_numpy(np.uint32, (n, rows)), want.view(np.uint32)), n


def test_wrapped_weights_at_any_float(ex):
    """A wrapped weight whose scales (Q8, Q4) or values (F32) start off a 16-byte
    boundary gives the aligned one's bits."""
    rng = oracle.RNG(4)
    rows, cols, n = 300, 512, 150
    dense = rng.fill_normal(rows * cols, 0.02).reshape(rows, cols)
    x = rng.fill_normal(n * cols, 1.0).reshape(n, cols)
    one = np.zeros(1, np.float32)
    for fmt in (srq.F32, srq.Q8, srq.Q4):
        w = srq.Weight.create(ex, dense, fmt)
        if fmt == srq.F32:
            vb, off = ex.upload(np.concatenate([one, dense.ravel().astype(np.float32)])), 4
            sp = None
        else:
            v, s = srq.pack(ex, dense, fmt)
            vb, off = ex.upload(v), 0
            sb = ex.upload(np.concatenate([one, np.asarray(s, np.float32).ravel()]))
            sp = C.c_void_p(sb.ptr.value + 4)
        h = C.c_void_p()
        srq.check(srq.lib().srq_weight_wrap(fmt, rows, cols, C.c_void_p(vb.ptr.value + off), sp, C.byref(h)))
        wrapped = srq.Weight(h)
        for m in (17, 32, n):  # (one row of such F32 values takes the generic GEMV, another order)
            print("wrapped", fmt, m, flush=True)
            got, want = srq.linear(ex, wrapped, x[:m]), srq.linear(ex, w, x[:m])
            assert np.array_equal(got.view(np.uint32), want.view(np.uint32)), (fmt, m)

"""The F32 GEMM's tiles and rings against FP64: 32- and 64-row tiles, K of one
step to more than the LDS ring holds, split and unsplit, ragged rows and
features, a row past the FP32 limit.  |err| <= (cols + 2) 2^-24 sum |x||w|: one
rounding per addition of the longest chain."""
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

"""Weights read by 128-byte row segments (calls of at most 32 rows): unrolled
slices of every length, slices run in chunks and slices that start inside a
segment, Q8 and Q4, against FP64 within (cols + 2) 2^-24 sum |x||w|, and rows
of 16- and 32-row tiles (a step's and a linear's) with the same bits as in a
call of 33 rows, which takes other tiles."""
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


@pytest.mark.parametrize("fmt", [srq.Q8, srq.Q4])
@pytest.mark.parametrize("rows,cols", [
    (9, 256),       # 4 blocks, fewer features than a tile
    (200, 1664),    # 26 blocks in slices of 5 (Q8 on odd blocks, Q4 inside segments)
    (8300, 832),    # 13 blocks, 256-feature tiles, the last block short
    (33000, 1152),  # 18 blocks, not split: two chunks of nine
    (33000, 1280),  # 20 blocks: two chunks of ten
    (16640, 3200),  # 50 blocks in slices of 17 (Q8: chunks that start on odd blocks), the last shorter
    (16500, 2176),  # 34 blocks in slices of 12, the last shorter
    (28672, 4096),  # slices of 32: two chunks of 16
    (4096, 14336),  # slices of 28: two chunks of 14
])
def test_segments(ex, fmt, rows, cols):
    rng = oracle.RNG(rows + cols)
    dense = np.resize(rng.fill_normal(1 << 18, 0.02), rows * cols).reshape(rows, cols)
    w = srq.Weight.create(ex, dense, fmt)
    x = np.resize(rng.fill_normal(1 << 16, 1.0), 33 * cols).reshape(33, cols).copy()
    x[20, 3] = 3e34
    want33 = srq.linear(ex, w, x)
    for n in (17, 31, 32):
        print("segments", fmt, rows, cols, n, flush=True)
        got = srq.linear(ex, w, x[:n])
        assert np.array_equal(got.view(np.uint32), want33[:n].view(np.uint32)), n
    some = np.unique(np.linspace(0, rows - 1, 40).astype(int))
    ow = oracle.Weight.from_dense(dense[some], oracle.Q8 if fmt == srq.Q8 else oracle.Q4)
    xd, wd = x.astype(np.float64), ow.dequant().astype(np.float64)
    bound = (cols + 2) * 2.0 ** -24 * (np.abs(xd) @ np.abs(wd).T)
    assert (np.abs(want33[:, some] - xd @ wd.T) <= bound).all()

"""The one-round GEMVs of short matrices (one row of at most 4096 columns): the
same bits as the streaming kernel, which a two-row call of the same row
takes, at the edges of their range -- one to four 1 KiB chunks, rows that end
inside a lane group, the most units and one more, a row past the FP32 limit."""
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
@pytest.mark.parametrize("rows,cols", [(1, 32), (3, 64), (577, 576), (2048, 1024), (960, 1056), (64, 2048), (4096, 96),
                                       (4097, 160), (1000, 2080), (9, 3072),
                                       (2050, 4064), (4096, 4096), (30, 4128),
                                       (3072, 256), (3073, 256), (4096, 256)])
def test_short_gemv(ex, fmt, rows, cols):
    rng = oracle.RNG(rows + cols)
    dense = rng.fill_normal(rows * cols, 0.02).reshape(rows, cols)
    w = srq.Weight.create(ex, dense, fmt)
    x = rng.fill_normal(2 * cols, 1.0).reshape(2, cols)
    for wide in (False, True):
        if wide:
            x[0, cols // 2] = -3e34
        print("short", fmt, rows, cols, wide, flush=True)
        got, want = srq.linear(ex, w, x[:1]), srq.linear(ex, w, x)
        assert np.array_equal(got[0].view(np.uint32), want[0].view(np.uint32))

"""The tall GEMM tiles (prefill chunks of Q8 / Q4 matrices): every output has
the bits of the same row in a call of at most 32 rows, which takes the small
tiles -- at the edges of row tiles (64 to 128 rows), of feature tiles (256 and
512), of K slices, for rows past the FP32 range and for matrices whose K is
not split; and srq_linear_noalloc, whose scratch may not hold the planes,
gives the same bits."""
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


def run(ex, entry, w, x):
    xb = ex.upload(np.ascontiguousarray(x, np.float32))
    yb = ex.empty(x.shape[0] * w.rows * 4)
    srq.check(getattr(srq.lib(), entry)(ex.h, yb.ptr, xb.ptr, w.h, x.shape[0]))
    ex.synchronize()
    return yb.to_numpy(np.float32, (x.shape[0], w.rows))


def small(ex, w, x):
    """The rows in calls of 17 to 32 rows (the last calls overlap)."""
    n, out = x.shape[0], np.empty((x.shape[0], w.rows), np.float32)
    for a in range(0, n, 32):
        a = min(a, n - 32)
        out[a:a + 32] = run(ex, "srq_linear", w, x[a:a + 32])
    return out


CASES = [
    # one row tile of every height, and its edges; one feature tile and a bit
    (srq.Q4, 516, 512, (33, 64, 65, 80, 81, 96, 97, 112, 113, 128, 129)),
    (srq.Q4, 7, 256, (33, 200)),            # fewer features than a wave, the shortest K
    (srq.Q4, 513, 256, (65, 129)),          # one feature in the last workgroup
    (srq.Q4, 32832, 256, (70, 300)),        # K not split: y written directly
    (srq.Q4, 2048, 3328, (160, 1024)),      # slices of 13 blocks, starting off the scale groups
    (srq.Q8, 2048, 8192, (193, 1024)),
    (srq.Q8, 4100, 1792, (200, 257, 700)),
    (srq.Q8, 33000, 768, (65, 129)),        # K not split
    (srq.Q8, 28672, 4096, (72, 130)),       # two slices
]


@pytest.mark.parametrize("fmt,rows,cols,ns", CASES)
def test_tall_tiles_match_small_tiles(ex, fmt, rows, cols, ns):
    rng = oracle.RNG(rows + cols)
    dense = np.resize(rng.fill_normal(1 << 20, 0.02), rows * cols).reshape(rows, cols)
    w = srq.Weight.create(ex, dense, fmt)
    for n in ns:
        x = rng.fill_normal(n * cols, 1.0).reshape(n, cols)
        x[n // 2, cols // 3] = 3e34  # past the FP32 limit of a row
        x[n - 1] = 0.0
        print("tall", fmt, rows, cols, n, flush=True)
        got, want = run(ex, "srq_linear", w, x), small(ex, w, x)
        assert np.array_equal(got.view(np.uint32), want.view(np.uint32)), n
        got = run(ex, "srq_linear_noalloc", w, x)
        assert np.array_equal(got.view(np.uint32), want.view(np.uint32)), n


@pytest.mark.parametrize("fmt,rows,cols", [(srq.Q4, 32832, 256), (srq.Q8, 33000, 768)])
@pytest.mark.parametrize("n", [66, 81, 128, 200])
def test_unsplit_wide_rows(ex, fmt, rows, cols, n):
    """Several rows past the FP32 limit in tiles that write y themselves, the
    first and last of a tile and those on either side of its 64th row."""
    rng = oracle.RNG(n)
    w = srq.Weight.create(ex, np.resize(rng.fill_normal(1 << 18, 0.02), rows * cols).reshape(rows, cols), fmt)
    x = rng.fill_normal(n * cols, 1.0).reshape(n, cols)
    x[[m for m in (0, 15, 63, 64, 79, 80, n - 1) if m < n], 7] = -3e34
    print("tall wide", fmt, rows, cols, n, flush=True)
    got, want = run(ex, "srq_linear", w, x), small(ex, w, x)
    assert np.array_equal(got.view(np.uint32), want.view(np.uint32))


@pytest.mark.parametrize("fmt,rows,cols,ns", [
    (srq.Q4, 516, 4096, (700,)),                 # 96 rows, split
    (srq.Q4, 1030, 3328, (600, 700)),            # 112 and 128 rows, split
    (srq.Q8, 12290, 768, (257,)),                # 96 rows, split
    (srq.Q8, 16384, 768, (129, 200)),            # 80 and 112 rows, split
    (srq.Q8, 4100, 1024, (800,)),                # 128 rows, split
    (srq.Q8, 33000, 256, (200, 257, 300)),       # 80, 96 and 112 rows, not split
    (srq.Q4, 33000, 256, (200, 257, 300)),
])
def test_tile_heights(ex, fmt, rows, cols, ns):
    """Each tile height that the choice between small and tall tiles leaves in
    use, for each format."""
    w = srq.Weight.create(ex, np.resize(oracle.RNG(rows).fill_normal(1 << 18, 0.02), rows * cols).reshape(rows, cols), fmt)
    for n in ns:
        print("tall heights", fmt, rows, cols, n, flush=True)
        x = np.resize(oracle.RNG(n).fill_normal(1 << 17, 1.0), n * cols).reshape(n, cols)
        got, want = run(ex, "srq_linear", w, x), small(ex, w, x)
        assert np.array_equal(got.view(np.uint32), want.view(np.uint32)), n

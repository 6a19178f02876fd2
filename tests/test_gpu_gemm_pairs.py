"""Weights read by 128-byte row segments (calls of at most 32 rows): unrolled
slices, slices run in chunks and slices that start inside a segment, Q8 and Q4,
against FP64 within (cols + 2) 2^-24 sum |x||w|, and rows of 32-row tiles with
the same bits as in a call of 33 rows, which takes other tiles; 16-row tiles,
which a step of 5 to 16 rows takes, with the bits of 17- to 33-row steps."""
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
    (8300, 832),    # 13 blocks, 256-feature tiles, the last block short (Q8: not by segments)
    (8300, 1664),   # 26 blocks in slices of 5, 256-feature tiles
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


@pytest.mark.parametrize("fmt", ["q8", "q4"])
@pytest.mark.parametrize("vocab,dim,heads,kv,hidden", [
    (33000, 1152, 9, 3, 512),    # head: 18 blocks, not split, 128-feature tiles
    (300, 4224, 33, 11, 4096),   # gate/up: 8192 features, slices of 17 blocks (odd starts), 64-feature tiles
    (300, 4608, 36, 6, 4096),    # gate/up: slices of 18 blocks
])
def test_16_row_tiles(ex, fmt, vocab, dim, heads, kv, hidden):
    """A session's logits in steps of 5 to 16 one-row sessions (16-row tiles) have
    the bits they have in steps of 17 and 32 (32-row tiles) and 33."""
    from sr_go_tranformer_amd import synthetic
    m = synthetic.build(ex, srq.make_config(vocab, dim, 1, heads, kv, hidden, 64, 10000.0, 1e-5, True), fmt, 7)
    pool = m.pool(33)
    ids = np.random.default_rng(dim).integers(0, vocab, 33)
    out = {}
    for n in (33, 32, 17, 16, 9, 5):
        print("16-row tiles", fmt, dim, n, flush=True)
        caches = [pool.cache(1) for _ in range(n)]
        for t in range(2):
            out[n] = m.step(caches, [[(int(i) + t) % vocab] for i in ids[:n]])
        for c in caches:
            c.close()
        assert np.isfinite(out[n]).all()
        assert np.array_equal(out[n].view(np.uint32), out[33][:n].view(np.uint32)), n

"""The one-round GEMVs of short matrices (one row of at most 4096 columns): the
same bits as the streaming kernel, which a two-row call of the same row
takes, at the edges of their range -- one to four 1 KiB chunks, rows that end
inside a lane group, the most units and one more, a row past the FP32 limit --
and, in decode steps, with the fused norm, bias, RoPE / KV write, residual and
SwiGLU."""
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


@pytest.mark.parametrize("fmt", ["q8", "q4"])
@pytest.mark.parametrize("dim,heads,kv,hidden", [
    (576, 9, 3, 1536),    # one chunk; down: two (Q8)
    (1600, 10, 2, 2048),  # two chunks (Q8), head size 160
    (2080, 13, 13, 2112), # eight waves a workgroup from here on, ragged last chunk
    (4096, 32, 8, 2304),  # the widest
])
def test_short_gemv_epilogues(ex, fmt, dim, heads, kv, hidden):
    """A session's logits after decode steps alone have the bits they have in
    steps of two and three sessions, whose layers take the streaming kernel."""
    from sr_go_tranformer_amd import synthetic
    cfg = srq.make_config(200, dim, 2, heads, kv, hidden, 64, 10000.0, 1e-5, True, qkv_bias=True)
    m = synthetic.build(ex, cfg, fmt, 11)
    rng = np.random.default_rng(dim)
    kd = dim // heads * kv
    for layer in range(2):
        for kind, n in ((srq.T_Q_BIAS, dim), (srq.T_K_BIAS, kd), (srq.T_V_BIAS, kd)):
            m.load(kind, layer, rng.normal(0, 0.3, n).astype(np.float32))
        for kind in (srq.T_ATTN_NORM, srq.T_FFN_NORM):
            m.load(kind, layer, rng.normal(1, 0.2, dim).astype(np.float32))
    prompt = [int(t) for t in rng.integers(0, 200, 6)]
    pool = m.pool(8)
    out = {}
    for n in (1, 2, 3):
        print("short epilogues", fmt, dim, n, flush=True)
        caches = [pool.cache(2) for _ in range(n)]
        for c in caches:
            m.step([c], [prompt])
        for t in range(3):
            out[n] = m.step(caches, [[7 + t + 5 * s] for s in range(n)], want=[True] + [False] * (n - 1))[0]
        for c in caches:
            c.close()
        assert np.isfinite(out[n]).all()
        assert np.array_equal(out[n].view(np.uint32), out[1].view(np.uint32)), n

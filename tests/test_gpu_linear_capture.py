"""srq_linear_enqueue in a captured graph: the graph of a matrix whose K is not
split holds no pointer into the executor's workspace, so replays stay right
after later calls have grown it, and other allocations keep their contents.
srq_linear_noalloc in a graph: right after other calls have used its array."""
import ctypes as C

import numpy as np
import pytest

import oracle
import sr_go_tranformer_amd as srq

pytestmark = pytest.mark.gpu

THREAD_LOCAL = 1  # hipStreamCaptureModeThreadLocal


@pytest.fixture(scope="module")
def ex():
    e = srq.Executor(0)
    yield e
    e.close()


@pytest.fixture(scope="module")
def hip():
    return C.CDLL("libamdhip64.so")


def capture(hip, ex, enqueue):
    stream, graph, run = C.c_void_p(ex.stream), C.c_void_p(), C.c_void_p()
    assert hip.hipStreamBeginCapture(stream, THREAD_LOCAL) == 0
    enqueue()
    assert hip.hipStreamEndCapture(stream, C.byref(graph)) == 0
    assert hip.hipGraphInstantiate(C.byref(run), graph, None, None, C.c_size_t(0)) == 0
    return run


def weight(ex, fmt, rows, cols, seed):
    return srq.Weight.create(ex, np.resize(oracle.RNG(seed).fill_normal(1 << 18, 0.02), rows * cols).reshape(rows, cols), fmt)


@pytest.mark.parametrize("entry,fmt,rows,cols,n", [
    ("srq_linear_enqueue", srq.Q4, 33000, 256, 70),    # unsplit, many rows
    ("srq_linear_enqueue", srq.Q8, 33000, 768, 130),
    ("srq_linear_enqueue", srq.Q8, 33000, 768, 24),
    ("srq_linear_enqueue", srq.Q4, 300, 512, 3),       # row by row
    ("srq_linear_noalloc", srq.Q4, 33000, 256, 70),
    ("srq_linear_noalloc", srq.Q4, 2048, 2048, 70),    # split: sums and planes in the fixed array
])
def test_replays_survive_workspace_growth(ex, hip, entry, fmt, rows, cols, n):
    print("capture", entry, fmt, rows, cols, n, flush=True)
    call = getattr(srq.lib(), entry)
    w = weight(ex, fmt, rows, cols, 3)
    x = ex.upload(oracle.RNG(4).fill_normal(n * cols, 1.0).reshape(n, cols))
    y = ex.empty(n * rows * 4)
    srq.check(call(ex.h, y.ptr, x.ptr, w.h, n))  # sizes whatever workspace the call uses
    ex.synchronize()
    want = y.to_numpy(np.uint32, (n, rows))
    run = capture(hip, ex, lambda: srq.check(call(ex.h, y.ptr, x.ptr, w.h, n)))
    big = weight(ex, srq.Q4, 4096, 4096, 5)
    for m in (200, 600, 1024):  # each larger call grows the workspace
        xm = oracle.RNG(m).fill_normal(m * 4096, 1.0).reshape(m, 4096)
        first = srq.linear(ex, big, xm)
        xb, yb = ex.upload(xm), ex.empty(m * 4096 * 4)
        srq.check(call(ex.h, yb.ptr, xb.ptr, big.h, m))  # the entry's own scratch, other contents
        ex.synchronize()
        pages = [ex.upload(np.full(1 << 18, k, np.uint32)) for k in range(32)]  # take what was given back
        y.write(np.zeros((n, rows), np.float32))
        assert hip.hipGraphLaunch(run, C.c_void_p(ex.stream)) == 0
        ex.synchronize()
        assert np.array_equal(y.to_numpy(np.uint32, (n, rows)), want), m
        assert all((p.to_numpy(np.uint32, (1 << 18,)) == k).all() for k, p in enumerate(pages)), m
        assert np.array_equal(srq.linear(ex, big, xm).view(np.uint32), first.view(np.uint32)), m
    assert hip.hipGraphExecDestroy(run) == 0

"""The packer's FP32 scale and rounding, against the oracle's FP64 division:
bit for bit, on whole-block rows (16-byte loads) and on odd widths and
unaligned sources (element loads)."""
import ctypes as C

import numpy as np
import pytest

import oracle
import sr_go_tranformer_amd as srq

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ex():
    return srq.Executor(0)


def near_ties(rows, cols, levels, seed):
    """Rows whose entries sit on half-integer multiples of their block's scale
    and one float to either side, over scales from the smallest the FP32 path
    takes to the largest, with subnormal, zero and huge blocks among them."""
    rng = np.random.default_rng(seed)
    groups = -(-cols // 64)
    out = np.zeros((rows, groups * 64), np.float32)
    for r in range(rows):
        for g in range(groups):
            e = [0, -8, -88, -91, 118, 121, -126, -140][(r + g) % 8]
            scale = (rng.uniform(1, 2) if (r // 8) % 2 else 1.0) * 2.0 ** e
            k = rng.integers(0, levels, 64) + 0.5
            v = np.minimum(k * scale, 3e38).astype(np.float32)
            side = rng.integers(0, 3, 64)
            v = np.where(side == 0, v, np.nextafter(v, np.float32(0) if r % 2 else np.float32(np.inf), dtype=np.float32))
            v[rng.integers(0, 64)] = np.float32(min(levels * scale, 3e38))
            v *= rng.choice(np.array([-1, 1], np.float32), 64)
            out[r, g * 64:(g + 1) * 64] = v
    out[3] = 0
    return np.ascontiguousarray(out[:, :cols])


@pytest.mark.parametrize("dtype", ["f32", "bf16", "f16"])
@pytest.mark.parametrize("fmt", ["q8", "q4"])
@pytest.mark.parametrize("rows,cols,offset", [(48, 64, 0), (33, 192, 0), (33, 192, 1), (40, 129, 0), (16, 7, 0), (65, 4096, 0)])
def test_pack_near_ties_bit_exact(ex, fmt, dtype, rows, cols, offset):
    print("pack near ties", fmt, dtype, rows, cols, offset, flush=True)
    f = near_ties(rows, cols, 127 if fmt == "q8" else 7, rows * cols)
    if dtype == "bf16":
        words = (f.view(np.uint32) >> 16).astype(np.uint16)
        f = (words.astype(np.uint32) << 16).view(np.float32)
    elif dtype == "f16":
        words = np.clip(f, -6e4, 6e4).astype(np.float16)
        f, words = words.astype(np.float32), words.view(np.uint16)
    else:
        words = f
    # `offset` elements in front leave the source unaligned
    src = ex.upload(np.concatenate([np.zeros(offset, words.dtype), words.ravel()]))
    F = {"q8": srq.Q8, "q4": srq.Q4}[fmt]
    vb, sb = srq.packed_bytes(F, rows, cols)
    v, s = ex.empty(vb), ex.empty(sb)
    D = {"f32": srq.SRC_F32, "bf16": srq.SRC_BF16, "f16": srq.SRC_F16}[dtype]
    srq.check(srq.lib().srq_pack(ex.h, F, rows, cols, C.c_void_p(src.value + offset * words.itemsize), D, v.ptr, s.ptr))
    ov, os_ = oracle.pack(f, oracle.Q8 if fmt == "q8" else oracle.Q4)
    assert np.array_equal(v.to_numpy(np.uint8, (vb,)), np.ascontiguousarray(ov).view(np.uint8).ravel())
    assert np.array_equal(s.to_numpy(np.uint32, (sb // 4,)), np.ascontiguousarray(os_).view(np.uint32).ravel())

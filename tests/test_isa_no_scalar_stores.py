"""The gfx950 code of every HIP source writes memory through vector
instructions only: each instruction of the compiler's assembly that stores,
is atomic, or writes back or discards cache lines is a vector or LDS one.

CPU-only: compiles each source with the library's own flags to assembly
(in parallel)."""
import concurrent.futures
import os
import re
import subprocess
import tempfile

import pytest

from sr_go_tranformer_amd import build as B

WRITES = re.compile(r"^\s+([a-z]\w*(?:store|write|atomic|_wb|discard)\w*)", re.M)
VECTOR = ("global_", "flat_", "buffer_", "scratch_", "ds_", "v_")
SOURCES = [s for s in B.SOURCES if s.endswith(".hip")]


def _assembly(src, tmp):
    out = os.path.join(tmp, src + ".s")
    cmd = [B.HIPCC, "-x", "hip", "--cuda-device-only", "-S"] + B.FLAGS + [
        "-I", os.path.join(B.HERE, "..", "include"), os.path.join(B.CSRC, src), "-o", out]
    r = subprocess.run(cmd, capture_output=True, text=True)
    assert r.returncode == 0, (src, r.stderr[-2000:])
    return src, open(out).read()


@pytest.mark.skipif(not os.path.exists(B.HIPCC), reason="hipcc not available")
def test_no_scalar_memory_writes():
    with tempfile.TemporaryDirectory() as tmp:
        with concurrent.futures.ThreadPoolExecutor(len(SOURCES)) as pool:
            results = list(pool.map(lambda s: _assembly(s, tmp), SOURCES))
    for src, asm in results:
        assert "gfx950" in asm, src
        seen = set(WRITES.findall(asm))
        assert not src.startswith("gemm") or any(m.startswith("global_store") for m in seen), (src, seen)
        assert all(m.startswith(VECTOR) for m in seen), (src, sorted(seen))

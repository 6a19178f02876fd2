"""The host-sanitized build compiles: the sources whose device code holds inline
asm, which its quick device compilation may reject, and the list of those it
compiles with optimisation is one of sources that exist."""
import os

import pytest

from sr_go_tranformer_amd import build as B

ASM = [s for s in B.SOURCES if s.endswith(".hip") and "lds_load" in open(os.path.join(B.CSRC, s)).read()]


def test_optimised_sources_exist():
    assert ASM and B.ASAN_O1 <= set(B.SOURCES)


@pytest.mark.skipif(not os.path.exists(B.HIPCC), reason="hipcc not available")
@pytest.mark.parametrize("src", ASM)
def test_sanitized_compile(src, tmp_path, monkeypatch):
    monkeypatch.setattr(B, "ASAN_DIR", str(tmp_path))
    assert os.path.getsize(B._compile_asan(src)) > 0

"""The bf16 tiles of the segmented products (csrc/seg_gemm.hip) through their own check program: every tile form at the edges of its rows, columns,
segments and k-tiles, bit for bit against the others and in samples against sums in double."""
import os
import subprocess

import pytest

EXE = os.path.join(os.path.dirname(os.path.abspath(__file__)), "cxx", "seg_tiles_check")


@pytest.mark.gpu
def test_tile_forms_give_the_same_bits():
    if not os.path.exists(EXE):
        pytest.fail("tests/cxx/seg_tiles_check is not built; run __graft_entry__.build()")
    r = subprocess.run([EXE], capture_output=True, text=True, timeout=110)
    print(r.stdout, r.stderr)
    assert r.returncode == 0, r.stdout + r.stderr
    assert " 0 failures" in r.stdout

"""The ordering check of the K-chunk fix-up (test_asm_ordering) on the matrix-core single-call kernel's unit, which
publishes its partial rows the same way. CPU only (hipcc cross-compiles)."""
import os
import subprocess

import pytest

from test_asm_ordering import CSRC, HIPCC, hipflags, unordered_publications


@pytest.mark.skipif(not os.path.exists(HIPCC), reason="hipcc not installed")
def test_mx_fixup_stores_complete_before_arrival(tmp_path):
    out = str(tmp_path / "mx.s")
    subprocess.run([HIPCC] + hipflags() + ["--cuda-device-only", "-S", os.path.join(CSRC, "p8x_gemv_mx.hip"), "-o", out], check=True,
                   stderr=subprocess.DEVNULL, timeout=600)
    n, bad = unordered_publications(open(out).read().splitlines())
    assert n > 0 and bad == 0, f"{bad} of {n} atomic adds follow an sc1 store without s_waitcnt vmcnt(0)"

"""The loops of the GEMM on split float32 operands: as generated, and with every register they write declared."""
import os
import subprocess
import sys

import pytest

from test_generated_asm import CSRC, _clobbers, _written_registers


@pytest.mark.parametrize("mode,inc", [("split128", "gemm_split_128_loop.inc"), ("split256x128", "gemm_split_256x128_loop.inc")])
def test_loop(mode, inc):
    out = subprocess.run([sys.executable, os.path.join(CSRC, "gen_gemm_asm.py"), mode], capture_output=True, text=True,
                         check=True).stdout
    text = open(os.path.join(CSRC, inc)).read()
    assert out == text and out.count("s_cbranch_scc1 L_loop_") == 1
    written = _written_registers(text)
    clob = _clobbers(open(os.path.join(CSRC, "gemm_split.hip")).read(), inc)
    assert "m0" in written and "scc" in clob and "memory" in clob
    assert written <= clob, sorted(written - clob)

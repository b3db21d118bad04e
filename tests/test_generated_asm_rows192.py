"""The loop of the 256 features x 192 tokens GEMM: as generated, and with every register it writes declared."""
import os
import subprocess
import sys

from test_generated_asm import CSRC, _clobbers, _written_registers


def test_loop():
    out = subprocess.run([sys.executable, os.path.join(CSRC, "gen_gemm_asm.py"), "rows192"], capture_output=True, text=True,
                         check=True).stdout
    text = open(os.path.join(CSRC, "gemm_bf16_256x192_loop.inc")).read()
    assert out == text and out.count("s_cbranch_scc1 L_loop_") == 1
    written = _written_registers(text)
    clob = _clobbers(open(os.path.join(CSRC, "gemm_bf16_256.hip")).read(), "gemm_bf16_256x192_loop.inc")
    assert "m0" in written and "scc" in clob and "memory" in clob
    assert written <= clob, sorted(written - clob)

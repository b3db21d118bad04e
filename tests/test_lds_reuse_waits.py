"""The key-split attention kernels reuse a wave's LDS space from round to round without a barrier: transposing reads of one
round, then the next round's memory-to-LDS loads into the same place.  The compiler does not order the two, so the source has
to wait for the reads.  Checked in the code generated for the device (no GPU needed)."""
import os
import re
import subprocess

import pytest

from cudabert_amd import build


@pytest.mark.parametrize("source,kernel,count", [("attention.hip", "attention_split_kernel", 1),
                                                 ("attention_f32.hip", "attention_f32_split_kernel", 2)])
def test_reads_are_waited_for_before_their_space_is_loaded_again(tmp_path, source, kernel, count):
    out = str(tmp_path / "k.s")
    subprocess.run([build.hipcc(), "-S", "--cuda-device-only", os.path.join(build.CSRC, source), "-o", out]
                   + build.COMMON_FLAGS + build.DEVICE_FLAGS, check=True, capture_output=True)
    bodies = re.findall(r"^_Z\w*%s\w*:.*?^\.Lfunc_end" % kernel, open(out).read(), re.S | re.M)
    assert len(bodies) == count
    for body in bodies:
        # the round is a loop whose blocks may be laid out rotated: what counts is the order around it
        events = re.findall(r"ds_read_b64_tr_b16|buffer_load_dword\w* [^\n]* lds|;;#ASMSTART(?:(?!;;#ASMEND).)*?s_waitcnt lgkmcnt\(0\)", body, re.S)
        kinds = "".join("W" if e.startswith(";;#ASM") else "L" if e.endswith("lds") else "R" for e in events)
        assert "R" in kinds and "L" in kinds
        assert "RL" not in kinds + kinds, kinds

"""The GEMMs that normalise in their epilogue fetch the residual from memory to LDS in pieces of four loads, wait for a piece by the
number of loads behind it and load its place again once it has been read.  Checked in the code generated for the device (no GPU
needed): reads are waited for before their place is loaded, every wait counts the loads that are there, and nothing else that the
counter counts (a store, a spilled register) comes between."""
import os
import re
import subprocess

import pytest

from cudabert_amd import build

EVENT = re.compile(r"ds_read\w*|buffer_load_dword\w* [^\n]* lds|(?:buffer|global|flat|scratch)_(?:store|load|atomic)\w*|s_waitcnt [^\n]*")


@pytest.fixture(scope="module")
def listing(tmp_path_factory):
    out = str(tmp_path_factory.mktemp("listing") / "k.s")
    subprocess.run([build.hipcc(), "-S", "--cuda-device-only", os.path.join(build.CSRC, "gemm_bf16_256.hip"), "-o", out]
                   + build.COMMON_FLAGS + build.DEVICE_FLAGS, check=True, capture_output=True)
    return open(out).read()


@pytest.mark.parametrize("kernel,columns", [(r"\d+gemm_bf16_t256_kernelILi0ELi6EE", 4), (r"\d+gemm_bf16_t256x192_ln_kernel", 3),
                                            (r"\d+gemm_bf16_t256x128_kernelILi0ELi6EE", 2)])
def test_residual_pieces(listing, kernel, columns):
    bodies = re.findall(r"^_Z\w*%s\w*:.*?; ScratchSize: \d+" % kernel, listing, re.S | re.M)
    assert len(bodies) == 1
    assert bodies[0].endswith("ScratchSize: 0")
    epilogue = bodies[0][bodies[0].rindex("v_mfma"):]
    events = EVENT.findall(epilogue[:re.search(r"s_waitcnt vmcnt\(0\)\n\s*;;#ASMEND(?![\s\S]*buffer_load_dword\w* [^\n]* lds)", epilogue).end()])
    events = events[next(i for i, e in enumerate(events) if e.endswith(" lds")):]
    loads, pieces, unread, last = 0, 0, False, 4 * columns
    for e in events:
        if e.endswith(" lds"):
            assert not unread, "a place is loaded again before its reads are waited for"
            loads += 1
        elif e.startswith("ds_read"):
            unread = True
        elif e.startswith("s_waitcnt"):
            unread = unread and "lgkmcnt(0)" not in e
            if "vmcnt" in e:
                left = int(re.search(r"vmcnt\((\d+)\)", e)[1])
                assert left == loads - 4 * (pieces + 1), (pieces, loads, left)
                pieces += 1
        else:
            pytest.fail("%s among the loads that are counted" % e)
    assert (loads, pieces) == (16 * columns, last)

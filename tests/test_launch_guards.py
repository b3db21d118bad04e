"""The launch switches of the bf16 GEMM kernels refuse an epilogue that has no kernel for the result type, instead of launching
another epilogue's: a small host program calls them past launch_gemm, whose own checks come first otherwise.  No GPU needed:
nothing may get as far as a launch."""
import os
import subprocess

import pytest

from cudabert_amd import build

PROGRAM = r"""
#include <cstdio>
#include "gemm_common.h"
namespace cubert {
bool launch_gemm_bf16_t256(const gemm_detail::GemmDev&, int, int, hipStream_t);
bool launch_gemm_bf16_t256x128(const gemm_detail::GemmDev&, int, int, hipStream_t);
bool launch_gemm_bf16_t256x128_deep(const gemm_detail::GemmDev&, int, int, hipStream_t);
bool launch_gemm_bf16_t128(const gemm_detail::GemmDev&, int, int, hipStream_t);
}
int main() {
    using namespace cubert;
    bool (*const launch[])(const gemm_detail::GemmDev&, int, int, hipStream_t) = {
        launch_gemm_bf16_t256, launch_gemm_bf16_t256x128, launch_gemm_bf16_t256x128_deep, launch_gemm_bf16_t128};
    const int refused[][2] = {{kBF16, kEpiBiasRes}, {kBF16, kEpiBiasResLN}, {kF32, kEpiBiasGeluUnits}, {kBF16, 99}, {kF32, 99}};
    for (auto f : launch)
        for (auto& r : refused) {
            gemm_detail::GemmDev d{};
            d.M = d.N = 256; d.K = d.ldx = 128; d.splits = d.tiles_n = d.tiles_m = 1;
            set_error("");
            const bool ok = f(d, r[0], r[1], nullptr);
            std::printf("%d %s\n", (int)ok, get_error());
        }
}
"""


@pytest.fixture(scope="module")
def lines(tmp_path_factory):
    from cudabert_amd import pybert                      # noqa: F401  (builds the library if there is none)
    d = tmp_path_factory.mktemp("guards")
    (d / "main.hip").write_text(PROGRAM)
    exe = str(d / "main")
    flags = build.COMMON_FLAGS + build.DEVICE_FLAGS
    for cmd in (["-c", str(d / "main.hip"), "-o", exe + ".o", "-I", build.CSRC] + flags,
                [exe + ".o", "-o", exe, build.LIB, "-Wl,-rpath," + build.HERE, "--hip-link"] + build.DEVICE_FLAGS):
        subprocess.run([build.hipcc()] + cmd, check=True, capture_output=True)
    return subprocess.run([exe], check=True, capture_output=True, text=True, env=dict(os.environ, HIP_VISIBLE_DEVICES="")).stdout.splitlines()


def test_an_epilogue_without_a_kernel_for_the_result_type_is_refused(lines):
    assert len(lines) == 20
    assert set(lines) == {"0 gemm: unknown epilogue"}, lines

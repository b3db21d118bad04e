"""The float32 GELU's two polynomials, on the host: against float64, interval by interval on both sides of zero, no further off than
x / 2 (1 + erf) with erf rounded correctly to float32.  No GPU needed."""
import numpy as np
import pytest

from host_program import compile_program, lines

PROGRAM = r"""
#include <cmath>
#include <cstdio>
#include <cstdlib>
#include <random>
#include "gemm_common.h"
using namespace cubert::gemm_detail;
int main(int argc, char** argv) {
    const double lo = std::atof(argv[1]), hi = std::atof(argv[2]);
    std::mt19937 r(1);
    std::uniform_real_distribution<double> u(lo, hi);
    double sq = 0, sq_ref = 0, most = 0, most_ref = 0;
    for (int i = 0; i < 200000; ++i) {
        const float x = (float)u(r), e = (float)std::exp2((double)(float)(x * x * -0.72134752044448170368f));
        const double want = 0.5 * x * std::erfc(-(double)x / std::sqrt(2.0));
        const float t = 1.0f + (float)std::erf((double)(x * 0.70710678118654752440f)), ref = x * 0.5f * t;
        const double d = std::fabs(gelu_with_exp(x, e) - want), d_ref = std::fabs(ref - want);
        sq += d * d; sq_ref += d_ref * d_ref;
        most = std::fmax(most, d); most_ref = std::fmax(most_ref, d_ref);
    }
    std::printf("%.9g %.9g %.9g %.9g\n", std::sqrt(sq / 200000), std::sqrt(sq_ref / 200000), most, most_ref);
}
"""
EDGES = [0.0, 0.01, 0.1, 0.25, 0.375, 0.5, 0.625, 0.75, 0.875, 1.0, 1.125, 1.25, 1.5, 2.0, 3.0, 4.0, 5.0, 5.5, 6.0, 8.0]


@pytest.fixture(scope="module")
def program(tmp_path_factory):
    return compile_program(PROGRAM, tmp_path_factory.mktemp("gelu"))


@pytest.mark.parametrize("sign", [-1, 1])
@pytest.mark.parametrize("lo,hi", list(zip(EDGES, EDGES[1:])))
def test_no_further_off_than_the_error_function(program, sign, lo, hi):
    rms, rms_ref, most, most_ref = map(float, lines(program, *sorted((sign * lo, sign * hi)))[0].split())
    assert rms <= rms_ref
    # the largest of 200 000: a rounding more where the two forms meet, next to one
    assert most <= most_ref * (1.2 if 0.875 <= lo < 1.25 else 1.0)
    assert np.isfinite(rms)

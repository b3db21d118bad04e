"""Parts that a pass is cut into, by the library's own rule at its default settings in bf16 mode."""
import pytest

from host_program import compile_program, lines

PROGRAM = r"""
#include <cstdio>
#include <cstdlib>
#include "engine.h"
int main(int argc, char** argv) {
    cubert::ModelOptions opt;
    opt.precision = cubert::kBF16;
    opt.split_keeps_one_round = true;
    opt.dims.hidden = std::atoi(argv[1]);
    opt.dims.inter = 4 * opt.dims.hidden;
    for (int i = 2; i < argc; ++i) std::printf("%d\n", cubert::Model::parts_of(opt, std::atol(argv[i]), 128));
}
"""


@pytest.fixture(scope="module")
def program(tmp_path_factory):
    return compile_program(PROGRAM, tmp_path_factory.mktemp("parts"))


def parts(program, hidden, rows):
    return list(map(int, lines(program, hidden, *rows)))


def test_two_rounds_on_an_xcd_are_no_reason_for_one_stream(program):
    """768 features: band b of 256 rows and its three workgroups belong to XCD b % 8, and 81 bands are 33 workgroups on one."""
    assert parts(program, 768, [14335, 14336, 20481, 20608, 21760, 21761]) == [1, 2, 2, 2, 2, 2]
    assert parts(program, 768, [20480]) == [1]


def test_one_round_of_1024_features(program):
    assert parts(program, 1024, [14335, 14336, 16384, 16385]) == [1, 1, 1, 2]

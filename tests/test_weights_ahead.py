"""Weights that LayerNorm and attention launches bring into the L2s: every line of the operand once, none outside it (the next
operand of the block, or nothing, lies there), for both layouts and widths that fill a last piece of 64 lines or leave it short.
No GPU needed."""
import pytest

from host_program import compile_program, lines

PROGRAM = r"""
#include <cstdio>
#include <cstdlib>
#include <set>
#include "l2_touch.h"
using namespace cubert;
template <bool SPLIT> void walk(int N, int K) {
    const size_t bytes = SPLIT ? split_bytes(N, K) : packed_bytes(N, (size_t)K * 2);
    const int groups = N / 32, n = l2_lines<SPLIT>(K), pieces = l2_pieces<SPLIT>(K);
    std::set<size_t> seen;
    size_t last = 0;
    for (int xcd = 0; xcd < 8; ++xcd)
        for (int g = groups * xcd / 8; g < groups * (xcd + 1) / 8; ++g)
            for (int line = 0; line < pieces * 64; ++line)
                if (line < n) { const size_t at = l2_offset<SPLIT>(K, g, line); seen.insert(at); last = at > last ? at : last; }
    const WeightsAhead a{reinterpret_cast<void*>(256), K, groups};
    std::printf("%zu %zu %d %zu %d\n", seen.size(), (size_t)groups * n, last + 128 <= bytes, (size_t)N * K * (SPLIT ? 6 : 2) / 128,
                l2_touch_workgroups<SPLIT>(a) % 8 + 8 * l2_touch_workgroups<SPLIT>(WeightsAhead()));
}
int main(int argc, char** argv) { std::atoi(argv[1]) ? walk<true>(std::atoi(argv[2]), std::atoi(argv[3])) : walk<false>(std::atoi(argv[2]), std::atoi(argv[3])); }
"""


@pytest.fixture(scope="module")
def program(tmp_path_factory):
    return compile_program(PROGRAM, tmp_path_factory.mktemp("ahead"))


@pytest.mark.parametrize("split_operands", [0, 1])
@pytest.mark.parametrize("N,K", [(32, 32), (96, 64), (768, 768), (3072, 1024), (1024, 4096), (2304, 160), (288, 1056)])
def test_every_line_once(program, split_operands, N, K):
    seen, touched, inside, operand, odd = map(int, lines(program, split_operands, N, K)[0].split())
    assert seen == touched == operand and inside == 1 and odd == 0

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


WALK = r"""
#include <cstdio>
#include <cstdlib>
#include <map>
#include "l2_touch.h"
using namespace cubert;
// argv: split operands, features, K, then  rows  or  heads batch query_blocks waves
template <bool SPLIT> void walk(int argc, char** argv) {
    const int N = std::atoi(argv[2]), K = std::atoi(argv[3]), groups = N / 32;
    const WeightsAhead a{reinterpret_cast<void*>(256), K, groups};
    std::map<size_t, int> seen;
    long wrong_xcd = 0;
    std::map<size_t, int> owner;
    for (int xcd = 0; xcd < 8; ++xcd)
        for (int g = groups * xcd / 8; g < groups * (xcd + 1) / 8; ++g)
            for (int line = 0; line < l2_lines<SPLIT>(K); ++line) owner[l2_offset<SPLIT>(K, g, line)] = xcd;
    auto wave = [&](const L2Share& s, int id) {
        for (int lane = 0; lane < 64; ++lane)
            l2_walk<SPLIT>(a, s, lane, [&](size_t at) { ++seen[at]; wrong_xcd += !owner.count(at) || owner[at] != (id & 7); });
    };
    if (argc == 5) {
        const int rows = std::atoi(argv[4]), grid = rows + l2_touch_workgroups<SPLIT>(a);
        for (int b = rows; b < grid; ++b)
            for (int w = 0; w < 4; ++w) wave(l2_share_after_rows(b, rows, grid, w), b);
    } else {
        const int heads = std::atoi(argv[4]), B = std::atoi(argv[5]), blocks = std::atoi(argv[6]), nw = std::atoi(argv[7]);
        const int gz = blocks + (l2_touch_workgroups<SPLIT>(a) / (nw / 4) + heads * B - 1) / (heads * B);
        for (int z = blocks; z < gz; ++z)
            for (int y = 0; y < B; ++y)
                for (int x = 0; x < heads; ++x)
                    for (int w = 0; w < nw; ++w) wave(l2_share_after_planes(x, y, z, heads, B, gz, blocks, nw, w), x + heads * (y + B * z));
    }
    long repeated = 0;
    for (auto& s : seen) repeated += s.second != 1;
    std::printf("%zu %zu %ld %ld\n", seen.size(), owner.size(), repeated, wrong_xcd);
}
int main(int argc, char** argv) { std::atoi(argv[1]) ? walk<true>(argc, argv) : walk<false>(argc, argv); }
"""


@pytest.fixture(scope="module")
def walk(tmp_path_factory):
    return compile_program(WALK, tmp_path_factory.mktemp("walk"))


@pytest.mark.parametrize("split_operands", [0, 1])
@pytest.mark.parametrize("N,K", [(32, 32), (96, 64), (768, 768), (4096, 1024), (288, 1056)])
@pytest.mark.parametrize("launch", [(1,), (17,), (128,), (4, 1, 1, 4), (12, 1, 1, 4), (12, 3, 5, 4), (16, 1, 7, 4), (1, 1, 1, 4), (3, 7, 2, 4), (16, 1, 4, 8), (12, 3, 1, 8)])
def test_launches_touch_every_line_once(walk, split_operands, N, K, launch):
    """What the workgroups added to a LayerNorm launch (rows) and to an attention launch (heads, lines, blocks of queries, waves of a workgroup) touch
    together, through the functions their kernels call: every line of the operand once, none outside it, each on the XCD whose tiles read it."""
    touched, operand, repeated, elsewhere = map(int, lines(walk, split_operands, N, K, *launch)[0].split())
    assert touched == operand and repeated == 0 and elsewhere == 0

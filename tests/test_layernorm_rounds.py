"""Tile of the GEMM that normalises in its epilogue: the smallest that leaves no CU with two workgroups, where a band of rows and
all its workgroups belong to one XCD of 32 CUs.  The launcher's choice against the workgroups each XCD gets, counted one by one."""
import pytest

from host_program import compile_program, lines

PROGRAM = r"""
#include <cstdio>
#include <cstdlib>
namespace cubert { int gemm_ln_pick_tile(int M, int N, int K, int elt); }
int main(int argc, char** argv) {
    for (int i = 2; i < argc; ++i) std::printf("%d\n", cubert::gemm_ln_pick_tile(std::atoi(argv[i]), std::atoi(argv[1]), 4 * std::atoi(argv[1]), 1));
}
"""
ROWS = {384: 128, 386: 192, 256: 256}         # tokens of the tile that a GemmParams::tile value names


@pytest.fixture(scope="module")
def program(tmp_path_factory):
    return compile_program(PROGRAM, tmp_path_factory.mktemp("rounds"))


def busiest_xcd(M, N, rows):
    """Workgroups on the XCD that gets most of them: ids go round the eight XCDs, XCD x walks the bands x, x + 8, ..."""
    bands, tiles_n, count = -(-M // rows), N // 256, [0] * 8
    for pid in range(8 * tiles_n * -(-bands // 8)):
        xcd, idx = pid % 8, pid // 8
        if idx // tiles_n * 8 + xcd < bands:
            count[xcd] += 1
    assert sum(count) == bands * tiles_n
    return max(count)


@pytest.mark.parametrize("N", [256, 512, 768, 1024])
def test_smallest_tile_of_one_round(program, N):
    Ms = sorted({6144, 70000} | {e + d for rows in (128, 192, 256) for bands in range(32, 300) for e in [bands * rows] for d in (0, 1)
                                 if 6144 <= e + d <= 70000})
    for M, tile in zip(Ms, map(int, lines(program, N, *Ms))):
        fits = [t for t in (384, 386) if busiest_xcd(M, N, ROWS[t]) <= 32]
        assert tile == (fits[0] if fits else 256), (M, N, tile, fits)


def test_few_rows_take_the_separate_kernels(program):
    assert lines(program, 768, 1, 6143, 6144) == ["0", "0", "384"]

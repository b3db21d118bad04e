"""Division as a multiplication and a shift, and the skinny kernel's tiles by it: every workgroup of a grid has a tile and a part of K of its own and
no tile is left out, also at row counts of several hundred thousand.  No GPU needed."""
import pytest

from host_program import compile_program, lines

PROGRAM = r"""
#include <cstdio>
#include <cstdlib>
#include <random>
#include <vector>
#include "gemm_skinny_map.h"
using namespace cubert::gemm_detail;
int divide() {
    int bad = 0;
    std::mt19937_64 r(1);
    auto check = [&](unsigned d, long x) {
        if (x < 0 || x >= 1L << 31) return;
        const Divisor v = divisor_of(d);
        bad += div_by((int)x, v.magic, v.shift) != (int)(x / d) || v.shift > 31;
    };
    for (int i = 0; i < 200000; ++i) {
        const unsigned d = i < 3000 ? i + 1 : 1 + (unsigned)(r() >> (33 + r() % 31)) % 0x7fffffffu;
        const long q = (0x7fffffffL / d);
        for (long k : {0L, 1L, q / 2, q - 1, q, (long)(r() % (q + 1))})
            for (long e : {-1L, 0L, 1L}) check(d, k * d + e);
        check(d, 0x7fffffffL);
        check(d, r() >> 33);
    }
    return bad;
}
int main(int argc, char** argv) {
    if (argc == 1) { std::printf("%d\n", divide()); return 0; }
    const int tiles_n = std::atoi(argv[1]), tiles_m = std::atoi(argv[2]), splits = std::atoi(argv[3]), cells = argc > 4 ? std::atoi(argv[4]) : 0;
    SkinnyMap m;
    if (!skinny_map(tiles_n, tiles_m, splits, cells, &m)) { std::printf("refused\n"); return 0; }
    std::vector<unsigned char> seen((size_t)tiles_n * tiles_m * splits);
    long outside = 0, twice = 0, idle = 0, elsewhere = 0;
    for (unsigned y = 0; y < m.grid_y; ++y)
        for (unsigned x = 0; x < m.grid_x; ++x) {
            int n, t, s;
            if (!skinny_tile(x, y, tiles_n, m.per_xcd, m.tiles_m, m.m_magic, m.split_magic, m.splits_more, m.shifts, &n, &t, &s)) { ++idle; continue; }
            if (n < 0 || n >= tiles_n || t < 0 || t >= tiles_m || s < 0 || s >= splits) { ++outside; continue; }
            if (cells) elsewhere += n / (tiles_n / cells) != (int)(x & 7) % cells || t / (tiles_m * cells / 8) != (int)(x & 7) / cells;
            twice += seen[((size_t)n * tiles_m + t) * splits + s]++;
        }
    long missing = 0;
    for (unsigned char c : seen) missing += !c;
    std::printf("%ld %ld %ld %ld %d\n", outside, twice, missing, elsewhere, (double)m.grid_x * 512 < 4294967296.0 && idle < 8L * splits + (m.grid_y > 1 ? (long)m.grid_x : 0));
}
"""


@pytest.fixture(scope="module")
def program(tmp_path_factory):
    return compile_program(PROGRAM, tmp_path_factory.mktemp("map"))


def test_division(program):
    assert lines(program) == ["0"]


# (features' tiles, tokens' tiles, parts): small grids that eight does not divide; 4096 features at 440 238 and 900 000 rows in 32 x 64 tiles, where a
# division that holds for x d < 2^32 puts tiles before the first row; more workgroups than a grid's x takes
@pytest.mark.parametrize("tiles_n,tiles_m,splits", [(1, 1, 1), (1, 3, 5), (7, 1, 3), (72, 1, 1), (128, 7, 2), (33, 25, 16), (128, 6879, 1), (128, 14063, 1),
                                                    (14, 18750, 3), (4, 125000, 1), (2, 262144, 255), (96, 70000, 1)])
def test_every_tile_once(program, tiles_n, tiles_m, splits):
    assert lines(program, tiles_n, tiles_m, splits) == ["0 0 0 0 1"]


@pytest.mark.parametrize("tiles_n,tiles_m,splits", [(4, 4, 1), (72, 8, 1), (96, 12, 4), (12, 20, 3)])
@pytest.mark.parametrize("cells", [2, 4])
def test_an_xcd_keeps_to_its_cell(program, tiles_n, tiles_m, splits, cells):
    assert lines(program, tiles_n, tiles_m, splits, cells) == ["0 0 0 0 1"]


def test_refused(program):
    assert lines(program, 1 << 20, 1 << 12, 1) == ["refused"]

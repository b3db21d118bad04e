"""Parts that a pass is cut into, by the library's own rule at its default settings in bf16 mode."""
import pytest

from host_program import compile_program, lines

PROGRAM = r"""
#include <cstdio>
#include <cstdlib>
#include "engine.h"
int main(int argc, char** argv) {
    cubert::ModelOptions opt;
    if (argc == 2) {
        opt.precision = std::atoi(argv[1]);
        cubert::read_split_options(&opt);
        std::printf("%d %d %d\n", opt.split_min_tokens, opt.split_parts, (int)opt.split_keeps_one_round);
        return 0;
    }
    opt.precision = cubert::kBF16;
    opt.split_keeps_one_round = true;
    opt.dims.hidden = std::atoi(argv[1]);
    opt.dims.inter = std::atoi(argv[2]);
    opt.fuse_residual = std::atoi(argv[3]);
    opt.fuse_layernorm = std::atoi(argv[4]);
    const bool waited = std::atoi(argv[5]);
    if (argc > 6 && std::atoi(argv[6]) == 0) {                    // a pass of parts of these rows
        std::vector<int> part_rows;
        for (int i = 7; i < argc; ++i) part_rows.push_back(std::atoi(argv[i]));
        std::printf("%d\n", cubert::Model::ln_tile_of_parts(opt, part_rows));
        return 0;
    }
    for (int i = 6; i < argc; ++i) {
        const long rows = std::atol(argv[i]);
        const int parts = cubert::Model::parts_of(opt, rows, 128, waited);
        std::vector<int> part_rows(parts, rows / parts);
        part_rows[0] += rows % parts;
        std::printf("%d %d", parts, cubert::Model::ln_tile_of_parts(opt, part_rows));
        for (long bits_of : {1000, 12000, 14336, 16000, 19000, 20000, 20480, 22000})
            std::printf(" %ld", cubert::Model::order_rows_of(opt, rows, bits_of, 128, waited));
        std::puts("");
    }
}
"""


@pytest.fixture(scope="module")
def program(tmp_path_factory):
    return compile_program(PROGRAM, tmp_path_factory.mktemp("parts"))


def plan(program, hidden, rows, inter=None, fuse_residual=1, fuse_layernorm=1, waited=1):
    """(parts, tile of the LayerNorm GEMMs that the pass prescribes) for every row count."""
    out = lines(program, hidden, inter or 4 * hidden, fuse_residual, fuse_layernorm, waited, *rows)
    return [tuple(map(int, l.split()[:2])) for l in out]


def parts(*args, **kw):
    return [p for p, _ in plan(*args, **kw)]


def test_two_rounds_on_an_xcd_are_no_reason_for_one_stream(program):
    """768 features: band b of 256 rows and its three workgroups belong to XCD b % 8, and 81 bands are 33 workgroups on one."""
    assert parts(program, 768, [14335, 14336, 20481, 20608, 21760, 21761]) == [1, 2, 2, 2, 2, 2]


def test_one_round_of_1024_features(program):
    """... while QKV and FFN-in have the tile of which a CU holds two, up to 15000 rows."""
    assert parts(program, 1024, [14335, 14336, 14976, 15104, 16384, 16385]) == [1, 1, 1, 2, 2, 2]


@pytest.mark.parametrize("without", [dict(fuse_residual=0), dict(fuse_layernorm=0), dict(inter=4128)])
def test_one_stream_asks_for_the_gemms_it_counts(program, without):
    """No residual or no LayerNorm in the epilogue, or an FFN-out (K not a multiple of 128) that does not have the 256 x 256 tile."""
    assert parts(program, 1024, [14336, 14976], **without) == [2, 2]


@pytest.mark.parametrize("hidden", [768, 1024])
def test_passes_that_queue_up_on_the_device_run_on_two_streams(program, hidden):
    assert parts(program, hidden, [14336, 16384, 18945, 20480], waited=0) == [2] * 4


@pytest.mark.parametrize("hidden", [256, 512, 768])
def test_narrow_models_run_on_two_streams(program, hidden):
    assert set(parts(program, hidden, range(14336, 70000, 256))) == {2}


@pytest.mark.parametrize("hidden,first,last", [(1024, 14336, 16384), (768, 18945, 20480)])
def test_parts_that_cover_the_chip_together_take_the_256_tile(program, hidden, first, last):
    rows = range(first + first % 2, last + 1, 14)
    assert set(plan(program, hidden, rows, waited=0)) == {(2, 256)}
    assert set(plan(program, hidden, rows)) == ({(1, 0), (2, 256)} if hidden == 1024 else {(2, 256)})
    beside = [14335, first - 1, last + 1, 25600, 32768]
    assert {t for _, t in plan(program, hidden, beside, waited=0)} == {0}
    assert {t for _, t in plan(program, hidden, rows, waited=0, fuse_layernorm=0)} == {0}


@pytest.mark.parametrize("hidden,part_rows,tile", [
    (1024, (8192, 8192), 256), (1024, (7937, 7937), 256), (1024, (8193, 7823), 386), (1024, (8769, 6683), 386),
    (768, (10240, 10240), 256), (768, (10241, 9629), 386), (768, (8752, 10317), 386), (768, (9618, 10687), 386),
    (768, (10753, 10753), 0), (1024, (8193, 8192), 0), (512, (16384, 16384), 0)])
def test_uneven_parts(program, hidden, part_rows, tile):
    """Bands are rounded up in each part: where the 256 x 256 workgroups of both parts are more than an XCD's 32, 256 x 192."""
    assert lines(program, hidden, 4 * hidden, 1, 1, 0, 0, *part_rows) == [str(tile)]
    xcd = sum(-(-(-(-n // 256)) // 8) * (hidden // 256) for n in part_rows)
    assert tile != 256 or xcd <= 32
    assert tile != 386 or xcd > 32


@pytest.mark.parametrize("hidden", [256, 768, 1024])
def test_a_pass_in_parts_regroups_no_sums(program, hidden):
    """Nor does one that gives the bits of a pass in parts."""
    rows, bits_of = [900, 11000, 14335, 14336, 15000, 18000, 18945, 20000], [1000, 12000, 14336, 16000, 19000, 20000, 20480, 22000]
    of = dict(zip(rows + bits_of, parts(program, hidden, rows + bits_of)))
    for n, l in zip(rows, lines(program, hidden, 4 * hidden, 1, 1, 1, *rows)):
        for padded, order in zip(bits_of, map(int, l.split()[2:])):
            assert order == (padded if of[n] == of[padded] == 1 else 0), (n, padded)


@pytest.mark.parametrize("precision,least", [(0, 8192), (1, 14336)])
def test_a_setting_of_the_default_value_changes_nothing(program, monkeypatch, precision, least):
    for name in ("MIN_TOKENS", "PARTS", "ONE_ROUND"):
        monkeypatch.delenv("CUBERT_SPLIT_" + name, raising=False)

    def options(**env):
        return tuple(map(int, lines(program, precision, **env)[0].split()))

    own = options()
    assert own == (least, 2, 1)
    assert own == options(CUBERT_SPLIT_MIN_TOKENS=str(least)) == options(CUBERT_SPLIT_PARTS="2") == options(CUBERT_SPLIT_ONE_ROUND="1") \
        == options(CUBERT_SPLIT_MIN_TOKENS="")
    assert options(CUBERT_SPLIT_ONE_ROUND="0") == (least, 2, 0)
    assert options(CUBERT_SPLIT_MIN_TOKENS="10000") == (10000, 2, 0)
    assert options(CUBERT_SPLIT_PARTS="3") == (least, 3, 0)

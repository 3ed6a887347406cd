"""The order in which gemm4w_tail_kernel adds up the parts of tail tiles (csrc/tail_units.h): every unit of a tile once, and the ones
that have rows spread over the XCDs (a block's index mod 8) whatever the number of rows."""
import ctypes
import subprocess

import pytest


@pytest.fixture(scope="module")
def units(tmp_path_factory):
    so = tmp_path_factory.mktemp("units") / "libtail_units.so"
    subprocess.check_call(["g++", "-O2", "-shared", "-fPIC", "-o", str(so), "tests/tail_units_host.cpp"])
    return ctypes.CDLL(str(so))


@pytest.fixture(scope="module")
def unit(units):
    def call(swiglu, item, wave, tile):
        out = (ctypes.c_int * 3)()
        units.t_tail_unit(int(swiglu), item, wave, tile, out)
        return tuple(out)
    return call


@pytest.mark.parametrize("swiglu", [False, True])
def test_every_unit_once(unit, swiglu):
    items, quarters = (16, 2) if swiglu else (32, 4)
    want = {(q, w, tt) for q in range(quarters) for w in range(4) for tt in range(8)}
    for tile in (0, 1, 7, 31, 250):
        got = [unit(swiglu, i, v, tile) for i in range(items) for v in range(4)]
        assert len(got) == len(want) and set(got) == want


@pytest.mark.parametrize("swiglu", [False, True])
@pytest.mark.parametrize("tiles", [8, 10, 40])
def test_units_with_rows_are_spread_over_the_xcds(unit, swiglu, tiles):
    items = 16 if swiglu else 32
    units = [(t, i, v, *unit(swiglu, i, v, t)) for t in range(tiles) for i in range(items) for v in range(4)]
    for rows in (1, 16, 17, 33, 64, 100, 128, 129, 200, 256):
        load = [0] * 8
        for t, i, _, _, w, tt in units:
            load[(t * items + i) % 8] += tt * 32 + (w >> 1) * 16 < rows
        # 16 rows of a tile are 8 units (4 for gate/up): with 8 tiles on 8 XCDs some unevenness is left
        assert min(load) > 0 and max(load) <= 2 * sum(load) / 8, (rows, load)


def test_blocks_of_a_part_are_the_ones_with_rows(units):
    for rows in range(1, 257):
        for w in range(4):
            assert units.t_part_blocks(rows, w) == sum(tt * 32 + (w >> 1) * 16 < rows for tt in range(8))


@pytest.mark.parametrize("tokens,want", [(300, 128), (450, 128), (475, 128), (482, 128), (484, 160), (500, 160), (512, 160)])
def test_height_of_a_layers_cut_tiles(units, tokens, want):
    """Four experts and a shared one in (2, 1) parts, 10 tiles along the features: three experts above 256 rows make 26 m-tiles of 128, one round
    of blocks and four more."""
    assert units.t_cut_height(128, 2 * tokens, 4, tokens, 2, 1, 10) == want
    if want > 128:
        over = [257, 257, 257, 2 * tokens - 771]
        assert sum(-(-c // want) * 2 for c in over) + -(-tokens // want) <= 25
    assert units.t_cut_height(256, 2 * tokens, 4, tokens, 2, 1, 10) == 256


def test_likely_tiles_are_no_more_than_the_rows_make(units):
    """Segments a standard deviation above the mean, against the most m-tiles of every division of the rows."""
    assert [units.t_likely_tiles(2 * t, 4, 256) for t in (470, 490, 512, 600, 1000, 1024)] == [4, 7, 7, 8, 11, 11]
    for rows, n, bm in ((9, 2, 4), (12, 3, 4), (13, 3, 4), (8, 4, 4), (2, 4, 4), (0, 3, 4), (17, 3, 8)):
        def divisions(left, k):
            return [(left,)] if k == 1 else [(a, *rest) for a in range(left + 1) for rest in divisions(left - a, k - 1)]
        most = max(sum(-(-c // bm) for c in d) for d in divisions(rows, n))
        mu = rows / n
        assert units.t_likely_tiles(rows, n, bm) == min(most, n * -(-int(mu + mu ** 0.5) // bm))

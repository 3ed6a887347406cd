"""How tiles of one or two lengths are dealt out to the blocks of the 4-wave kernel (csrc/tail_units.h, g4_place): every tile once, a block's items
without gaps, long ones first, and blocks without a long one of the last round ahead by `light_rounds` short ones."""
import ctypes
import random
import subprocess

import pytest


@pytest.fixture(scope="module")
def place(tmp_path_factory):
    so = tmp_path_factory.mktemp("place") / "libplace.so"
    subprocess.check_call(["g++", "-O2", "-shared", "-fPIC", "-o", str(so), "tests/tail_units_host.cpp"])
    return ctypes.CDLL(str(so)).t_place


CASES = [(0, 0, 0), (1, 0, 0), (80, 0, 0), (256, 0, 0), (257, 1, 1), (340, 160, 1), (330, 171, 2), (440, 220, 1), (512, 300, 0), (10, 700, 3), (240, 15, 1)]


@pytest.mark.parametrize("longs,shorts,light_rounds", CASES + [
    (r.randrange(1200), r.randrange(800), r.randrange(4)) for r in [random.Random(5)] for _ in range(40)])
def test_every_tile_once(place, longs, shorts, light_rounds):
    if longs % 256 == 0:
        light_rounds = 0
    seen = []
    for xcd in range(8):
        for slot in range(32):
            items = [place(longs, shorts, light_rounds, xcd, slot, i) for i in range(16)]
            there = [v for v in items if v >= 0]
            assert items == there + [-1] * (16 - len(there))
            kinds = [v & 1 for v in there]
            assert kinds == sorted(kinds)
            n_long = kinds.count(0)
            assert n_long in (longs // 256, -(-longs // 256))
            if n_long == longs // 256 and longs % 256 and shorts >= light_rounds * (256 - longs % 256):
                assert kinds.count(1) >= light_rounds
            seen += there
    assert sorted(seen) == sorted([2 * t for t in range(longs)] + [2 * t + 1 for t in range(shorts)])


def test_a_last_round_is_spread_over_the_xcds(place):
    for left in (8, 80, 129, 250):
        per_xcd = [sum(place(256 + left, 0, 0, xcd, slot, 1) >= 0 for slot in range(32)) for xcd in range(8)]
        assert sum(per_xcd) == left and max(per_xcd) == -(-left // 8)

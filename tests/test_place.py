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


def heights(rows, cap):
    blocks = -(-rows // 32)
    mt = -(-blocks // cap)
    return mt, max(4, -(-blocks // mt)) if mt else 4


@pytest.mark.parametrize("seed", range(60))
def test_the_longest_block_is_what_the_model_says(place, seed):
    """csrc/gemm4w.h, g4_two_lengths, against the blocks that g4_place fills: long tiles from the highest to the lowest, short ones priced alike."""
    from comfyui_amd import _lib
    PAIR = {4: 58, 5: 70, 6: 80, 7: 90, 8: 100}
    rng = random.Random(seed)
    E, N = rng.choice([2, 4, 8, 16]), 256 * rng.choice([2, 8, 10])
    K, Ks = rng.choice([(6912, 3584), (3584, 6912), (2560, 512), (512, 1024)])
    T = rng.randint(300, 5000)
    cuts = sorted(rng.randint(0, 2 * T) for _ in range(E - 1))
    rows = [b - a for a, b in zip([0] + cuts, cuts + [2 * T])]
    for cap_long, cap_short in ((8, 8), (4, 4), (5, 8), (7, 6)):
        rounds = ctypes.c_int()
        got = _lib.lib.hdmoe_two_lengths(E, (ctypes.c_int * E)(*rows), K, T, Ks, N, cap_long, cap_short, ctypes.byref(rounds))
        groups = [(r, K) for r in rows] + [(T, Ks)]
        kl, ks = max(K, Ks), min(K, Ks)
        tiles = {k: sorted((h for r, kk in groups if kk == k for mt, h in [heights(r, cap_long if k == kl else cap_short)] for _ in range(mt * N // 256)),
                           reverse=True) for k in (kl, ks)}
        price = lambda k, h: k // 256 * PAIR[h] + 150
        short = price(ks, tiles[ks][0])
        longest = 0
        for xcd in range(8):
            for slot in range(32):
                cost, i = 0, 0
                while (v := place(len(tiles[kl]), len(tiles[ks]), rounds.value, xcd, slot, i)) >= 0:
                    # a round of long tiles takes what its first one does
                    cost, i = cost + (short if v & 1 else price(kl, tiles[kl][(v >> 1) // 256 * 256])), i + 1
                longest = max(longest, cost)
        assert got == longest, (rows, T, K, Ks, N, cap_long, cap_short)


@pytest.mark.parametrize("lists", [[60, 60, 30, 60, 40], [30] * 5, [0, 1, 0, 7, 9], [250], [20] * 12, [40, 40, 40, 40, 20]] + [
    [r.randrange(90) for _ in range(r.randrange(1, 17))] for r in [random.Random(9)] for _ in range(30)])
def test_lists_are_dealt_out_evenly(tmp_path_factory, place, lists):
    """csrc/tail_units.h, g4_dealt: each list in contiguous shares, no XCD more than one tile ahead in a list or in all of them, and a round of
    256 blocks takes whatever has 256 tiles."""
    so = next(tmp_path_factory.getbasetemp().glob("place*")) / "libplace.so"
    dealt = ctypes.CDLL(str(so)).t_dealt
    ends = [sum(lists[:k]) for k in range(len(lists) + 1)]
    load = [0] * 8
    for a, b in zip(ends, ends[1:]):
        cuts = [dealt(b, x) - dealt(a, x) for x in range(9)]
        assert cuts[0] == 0 and cuts[8] == b - a
        shares = [cuts[x + 1] - cuts[x] for x in range(8)]
        assert min(shares) >= (b - a) // 8 and max(shares) <= -(-(b - a) // 8)
        load = [l + v for l, v in zip(load, shares)]
    assert max(load) - min(load) <= 1 and max(load) == -(-ends[-1] // 8)

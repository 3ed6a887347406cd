"""The cut of tail tiles along K (csrc/gemm4w.h, g4_plan_tail) against its cost model in exact arithmetic. The kernel that leaves
the parts and the one that adds them up each work the plan out; it must not depend on how a compiler rounds."""
import ctypes
import random
from fractions import Fraction

import pytest

from comfyui_amd import _lib

CUS = 256


def plan(code, tiles, K, padding):
    rounds, left = ctypes.c_int(-1), ctypes.c_int(-1)
    parts = _lib.lib.hdmoe_tail_plan(code, tiles, K, padding, ctypes.byref(rounds), ctypes.byref(left))
    return rounds.value, left.value, parts


def exact(code, tiles, K, padding):
    """The cheapest number of parts: pairs of K steps of the longest part, 4.5 for the second launch, 0.04 per part of a full tile,
    against 0.85 of the uncut tile's pairs; the average tile's rows in whole rows."""
    left, pairs = tiles % CUS, K // 128
    fill = Fraction(256 - padding // tiles, 256)
    best, parts = Fraction(85, 100) * pairs, 1
    for p in range(2, 13):
        if left == 0 or p * left > CUS or pairs // p < (3 if code == _lib.W_E4M3FN_UPCAST else 2):
            break
        cost = -(-pairs // p) + Fraction(9, 2) + Fraction(4, 100) * fill * p * left
        if cost < best:
            best, parts = cost, p
    return tiles // CUS, left, parts


@pytest.mark.parametrize("code", [_lib.W_BF16, _lib.W_E4M3FN_UPCAST])
def test_plan_is_the_cost_model_to_the_last_digit(code):
    rng = random.Random(code)
    cuts = set()
    for _ in range(20000):
        tiles = rng.choice([rng.randint(1, 300), rng.randint(1, 6000)])
        K = 128 * rng.choice([rng.randint(1, 60), rng.randint(1, 300)])
        padding = rng.choice([0, rng.randint(0, 255 * tiles)])
        got = plan(code, tiles, K, padding)
        assert got == exact(code, tiles, K, padding), (tiles, K, padding)
        cuts.add(got[2])
    assert cuts >= set(range(1, 9))


def test_rounds_and_tiles_left_over():
    # 10 pairs: 2 parts of 25 tiles cost 5 + 4.5 + 2 > 8.5, in the first round as in a later one
    assert plan(_lib.W_BF16, 25, 1280, 0) == (0, 25, 1) and plan(_lib.W_BF16, 3 * CUS + 25, 1280, 0) == (3, 25, 1)
    assert plan(_lib.W_BF16, 2 * CUS, 2560, 0) == (2, 0, 1)


def test_sizes_out_of_range():
    for args in [(0, 2560, 0), (5, 0, 0), (5, 2560, -1), (5, 2560, 5 * 256), (5, 128 * 40000, 0)]:
        assert plan(_lib.W_BF16, *args)[2] == 0

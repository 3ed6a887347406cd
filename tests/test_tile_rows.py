"""The height of the tiles of a Linear (csrc/gemm4w.h, g4_best_cap) against its cost model written out: rounds over 256 CUs, the
highest tiles first, a pair of K steps priced by the height of the round's first tile."""
import random

import pytest

from comfyui_amd import _lib

CUS = 256
PAIR = {4: 58, 5: 70, 6: 80, 7: 90, 8: 100}


def tile_rows(code, rows, K, N):
    return _lib.lib.hdmoe_linear_tile_rows(code, rows, K, N)


def model(code, rows, K, N):
    pairs, nt = K // 128, N // 256
    tiles = -(-rows // 256) * nt
    parts = _lib.lib.hdmoe_tail_plan(code, tiles, K, (-rows % 256) * nt, None, None)
    if tiles > 24 * CUS:
        parts = 1
    whole = -(-tiles // CUS)
    if parts > 1:
        return 256
    if rows <= 128 and code != _lib.W_E4M3FN_UPCAST:
        return 0
    best, limit = 8, whole * (100 * pairs + 150)
    limit -= limit // 12
    blocks = -(-rows // 32)
    for cap in (8, 7, 6, 5, 4):
        mt = -(-blocks // cap)
        height = max(4, -(-blocks // mt))
        cost = -(-mt * nt // CUS) * (pairs * PAIR[height] + 150)
        if whole <= 24 and cost < limit:
            best, limit = height, cost
    return 32 * best


@pytest.mark.parametrize("code", [_lib.W_BF16, _lib.W_F16, _lib.W_E4M3FN_UPCAST])
def test_heights_are_the_cost_model(code):
    rng = random.Random(code)
    seen = set()
    for _ in range(20000):
        rows = int(2 ** rng.uniform(0, 16))
        K = 128 * rng.choice([rng.randint(3, 40), rng.randint(3, 120)])
        N = 256 * rng.randint(1, 40)
        got = tile_rows(code, rows, K, N)
        assert got == model(code, rows, K, N), (rows, K, N)
        seen.add(got)
    assert seen >= {128, 160, 192, 224, 256}


def test_sizes_out_of_range():
    assert tile_rows(_lib.W_E4M3FN, 1000, 2560, 2560) == 0          # fp8 activations
    assert tile_rows(_lib.W_E4M3FN_UPCAST, 1000, 256, 2560) == 0
    assert tile_rows(_lib.W_BF16, 1000, 2624, 2560) == 0
    assert tile_rows(_lib.W_BF16, 1000, 2560, 2500) == 0
    assert tile_rows(_lib.W_BF16, 0, 2560, 2560) == 0


def test_fp8_heights_are_the_cost_model():
    """No tile is cut, and without a cap a tile is as high as its rows need."""
    rng = random.Random(8)
    seen = set()
    for _ in range(20000):
        rows = int(2 ** rng.uniform(0, 16))
        K = 256 * rng.choice([rng.randint(2, 20), rng.randint(2, 60)])
        N = 256 * rng.randint(1, 40)
        pairs, nt, blocks = K // 256, N // 256, -(-rows // 32)
        whole = -(-(-(-rows // 256) * nt) // CUS)
        want, limit = max(4, min(8, blocks)), whole * (100 * pairs + 150)
        limit -= limit // 12
        for cap in (8, 7, 6, 5, 4):
            mt = -(-blocks // cap)
            height = max(4, -(-blocks // mt))
            cost = -(-mt * nt // CUS) * (pairs * PAIR[height] + 150)
            if whole <= 24 and cost < limit:
                want, limit = height, cost
        got = _lib.lib.hdmoe_fp8_linear_tile_rows(rows, K, N)
        assert got == 32 * want, (rows, K, N)
        seen.add(got)
    assert seen == {128, 160, 192, 224, 256}
    for bad in ((0, 2560, 2560), (1000, 384, 2560), (1000, 256, 2560), (1000, 2560, 2500)):
        assert _lib.lib.hdmoe_fp8_linear_tile_rows(*bad) == 0

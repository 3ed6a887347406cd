"""The tiles of the fp8 gate/up kernel on 224 and 128 tokens (csrc/swiglu224.h, csrc/tail_units.h): every style covers a segment's rows once, each block
walks its high tiles before its low ones, and the longest block is what the cost that picks a style says."""
import ctypes
import random
import subprocess

import pytest

STYLES, HIGH, LOW = 5, 100, 75


@pytest.fixture(scope="module")
def lib(tmp_path_factory):
    so = tmp_path_factory.mktemp("s224") / "libs224.so"
    subprocess.check_call(["g++", "-O2", "-shared", "-fPIC", "-o", str(so), "tests/tail_units_host.cpp"])
    return ctypes.CDLL(str(so))


def mix(lib, rows, style):
    v = lib.t_mix(rows, style)
    return v & 0xffff, v >> 16


@pytest.mark.parametrize("style", range(STYLES))
def test_a_segment_is_covered(lib, style):
    for rows in [*range(0, 1000), 2047, 2048, 2049, 4096, 32768]:
        highs, lows = mix(lib, rows, style)
        room = 224 * highs + 128 * lows
        assert rows <= room
        if lows:
            assert 224 * highs + 128 * (lows - 1) < rows     # none without rows
        elif highs:
            assert 224 * (highs - 1) < rows
        else:
            assert rows == 0


def block_tiles(lib, highs, lows, xcd, slot):
    """What the kernel's table holds for a block: ('h' | 'l', index in the list of that kind)."""
    rounds, left = divmod(highs, 256)
    out = [("h", xcd * rounds * 32 + slot + 32 * i) for i in range(rounds)]
    for i in range(64):
        v = lib.t_place(left, lows, 1 if left else 0, xcd, slot, i)
        if v < 0:
            return out
        out.append(("l", v >> 1) if v & 1 else ("h", rounds * 256 + (v >> 1)))
    raise AssertionError


@pytest.mark.parametrize("highs,lows", [(0, 0), (1, 0), (0, 1), (256, 0), (256, 1), (244, 28), (272, 0), (0, 544), (56, 460), (2448, 244), (4896, 244)] + [
    (r.randrange(1500), r.randrange(900)) for r in [random.Random(3)] for _ in range(30)])
def test_every_tile_once_high_ones_first(lib, highs, lows):
    seen, longest = [], 0
    for xcd in range(8):
        for slot in range(32):
            mine = block_tiles(lib, highs, lows, xcd, slot)
            kinds = [k for k, _ in mine]
            assert kinds == sorted(kinds)
            longest = max(longest, kinds.count("h") * HIGH + kinds.count("l") * LOW)
            seen += mine
    assert sorted(seen) == [("h", i) for i in range(highs)] + [("l", i) for i in range(lows)]
    assert longest == lib.t_s224_cost(highs, lows)

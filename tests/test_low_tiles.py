"""Where fp8 gate/up contractions take low tiles and the kernel on 224-token tiles (csrc/tail_units.h, s224_price; csrc/gemm.hip, s224_pays): a low tile
behind high ones of the same weights reads them from memory again."""
import ctypes
import subprocess

import pytest

from comfyui_amd import _lib

H, HS = 54, 28   # columns of a hidden width of 6912 and 3584


@pytest.fixture(scope="module")
def lib(tmp_path_factory):
    so = tmp_path_factory.mktemp("mix") / "libmix.so"
    subprocess.check_call(["g++", "-O2", "-shared", "-fPIC", "-o", str(so), "tests/mix_host.cpp"])
    return ctypes.CDLL(str(so))


def styles(lib, segments, shared, cols=H, shared_cols=HS, width=2560):
    rows, n = [*segments, shared], len(segments) + 1
    arr = lambda v: (ctypes.c_int * n)(*v)
    return divmod(lib.t_style(n, 1, arr(rows), arr([cols] * (n - 1) + [shared_cols]), width), 5)


@pytest.mark.parametrize("experts,tokens,width", [(16, 2048, 2560), (16, 2400, 2560), (16, 1800, 2560), (12, 1600, 2560), (12, 1800, 2560), (8, 1024, 2560),
                                                  (8, 2200, 2560), (6, 850, 2560), (4, 1000, 4096), (4, 640, 4096)])
def test_no_low_tile_of_an_expert_behind_a_high_one(lib, experts, tokens, width):
    """Measured 4 to 12 % slower than high tiles alone: what a round of tiles costs less, the weights read twice cost more."""
    mean, sd = 2 * tokens / experts, (2 * tokens / experts * (1 - 2 / experts)) ** 0.5
    for off in (0, 0.5, 1):
        segments = [round(mean + (off * sd if e % 2 else -off * sd)) for e in range(experts)]
        of_experts, _ = styles(lib, segments, tokens, *((H, HS) if width == 2560 else (86, 44)), width)
        assert of_experts in (0, 3, 4), (segments, of_experts)   # high ones alone, or lows that share their weights among themselves


@pytest.mark.parametrize("tokens", [350, 400, 560, 700, 768, 850, 1024])
def test_low_tiles_that_end_a_round(lib, tokens):
    """The layer's own sizes, where they gain 4 to 14 %."""
    assert styles(lib, [tokens // 2 + d for d in (-8, 8, -8, 8)], tokens) != (0, 0)


@pytest.mark.parametrize("rows,low", [(128, False), (256, True), (257, True), (400, True), (513, False), (1024, False), (1300, True), (1500, True), (2000, False)])
def test_low_tiles_on_16_bit_activations(lib, rows, low):
    """A dense feed-forward of 6912 features on 256-row tiles."""
    assert (lib.t_style16(rows, H, 27) != 0) == low


def test_price(lib):
    assert lib.t_price(432, 0, 0, 4) == 200 and lib.t_price(432, 32, 0, 4) == 202   # beside the last round's high tiles
    assert lib.t_price(1144, 864, 864, 4) > lib.t_price(2008, 0, 0, 4)
    assert lib.t_shift(86, 4096, 1) == 5 and lib.t_shift(244, 2560, 2047) == 4 and lib.t_shift(244, 2560, 2048) == 8 and lib.t_shift(1 << 20, 1 << 20, 4096) == 4


def name(tokens, experts, d=2560, h=6912, hs=3584, scaled=1):
    return _lib.lib.hdmoe_gate_up_kernel_name(_lib.W_E4M3FN, tokens, experts, d, h, hs, scaled)


@pytest.mark.parametrize("scaled", [0, 1])
def test_where_the_kernel_runs(scaled):
    """Layers and dense branches at both sides of the lines (dense: 256 stands for the width of experts that there are none of)."""
    is224 = lambda *a, **k: name(*a, **k, scaled=scaled) == b"swiglu224_kernel"
    dense = lambda rows, d=2560, h=6912: is224(rows, 0, d, 256, h)
    for tokens in (257, 300, 320):
        assert not is224(tokens, 4)
    for tokens in [321, 448, 491, 513, 768, 1024, 1300, 2400, 4096, 8192]:
        assert is224(tokens, 4)
    for tokens, takes in ((257, True), (448, True), (449, False), (512, False), (513, True), (2048, True)):
        assert is224(tokens, 8) == takes
    for rows, takes in ((385, True), (512, True), (513, False), (577, False), (768, False), (769, True), (896, True), (897, False), (1024, False),
                        (1025, False), (1280, False), (1281, True), (2048, True), (2049, False), (2304, False), (2305, True), (3584, True), (4480, True), (8192, True)):
        assert dense(rows) == takes, rows
    assert not dense(449, h=32768) and not dense(480, h=32768) and dense(513, h=32768)
    assert not dense(640, 4096, 11008) and dense(641, 4096, 11008)

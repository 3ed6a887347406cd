"""The cut along K of a dense fp8 down projection (csrc/gemm.hip, hdmoe_down_parts), as the working memory shows it."""
import pytest

from comfyui_amd import _lib

D, H = 2560, 6912


def parts(rows, dim=D, hidden=H):
    align = lambda n: -(-n // 256) * 256
    room = _lib.lib.hdmoe_ffn_workspace_bytes(rows, dim, hidden, _lib.W_E4M3FN) - align(rows * dim) - align(rows * hidden)
    assert room % (rows * dim * 4) < 256 or room % (rows * dim * 4) == 0
    return room // (rows * dim * 4) or 1


@pytest.mark.parametrize("rows,want", [(300, 6), (512, 4), (768, 3), (1024, 3), (1280, 2), (1536, 2), (1600, 2), (1700, 2), (1900, 2), (2048, 2), (2560, 1), (4096, 1)])
def test_parts(rows, want):
    """Whole tiles take their K steps one after the other while cold weights arrive: two parts up to 2048 rows."""
    assert parts(rows) == want


@pytest.mark.parametrize("rows,want", [(1536, 2), (1537, 2), (1700, 2), (1793, 1)])
def test_parts_on_tiles_of_any_height(rows, want):
    """At width 4096 only 224- and 256-token tiles in two parts fit a round there; whole ones on 128-token tiles wait for cold weights."""
    assert parts(rows, 4096, 11008) == want


def test_few_steps_are_not_cut():
    assert parts(1700, 512, 1280) == 1   # 5 pairs of K steps: no part has three


@pytest.mark.parametrize("tokens", [1100, 2049, 2051, 2100, 2300, 2560, 2561, 4096, 8192])
def test_whole_tiles_run_on_the_4_wave_kernel(tokens):
    name = _lib.lib.hdmoe_plain_kernel_name(2 * tokens, 4, H, tokens, 3584, D, 1, 0)
    assert name == b"gemm4w_kernel<F8, PLAIN>"


def layer_parts(tokens, dim, h, hs, experts=4):
    from comfyui_amd import functional as HF
    lay = HF.layer_layout(tokens, dim, h, hs, experts, _lib.W_E4M3FN)
    return (lay.flags - lay.partials) // (3 * tokens * dim * 4) or 1


@pytest.mark.parametrize("dim,h,hs,tokens,want", [(2560, 6912, 3584, 512, 2), (2560, 6912, 3584, 960, 2), (2560, 6912, 3584, 1024, 1), (4096, 11008, 5632, 470, 3),
                                                  (4096, 11008, 5632, 490, 2), (4096, 11008, 5632, 512, 2), (4096, 11008, 5632, 520, 1)])
def test_parts_of_a_layer(dim, h, hs, tokens, want):
    """Four experts of just under 256 rows make 7 tiles of 256 rows at most, not 8: two parts fit a round at width 4096."""
    assert layer_parts(tokens, dim, h, hs) == want


def few_rows_partials(tokens, code, dim=2560, h=6912, hs=3584, experts=4):
    from comfyui_amd import functional as HF
    lay = HF.layer_layout(tokens, dim, h, hs, experts, code)
    return (lay.flags - lay.partials) // (3 * tokens * dim * 4) or 1


@pytest.mark.parametrize("code", [_lib.W_E4M3FN, _lib.W_BF16, _lib.W_E4M3FN_UPCAST])
@pytest.mark.parametrize("tokens,parts,shared", [(1, 6, 4), (16, 5, 3), (64, 5, 3), (128, 5, 3), (129, 4, 2), (130, 3, 2), (256, 3, 2)])
def test_parts_of_few_rows_fit_a_round_however_they_are_routed(code, tokens, parts, shared):
    """Every division of the slots that no token's two experts rule out, in 128-token tiles by 10 along the features."""
    assert few_rows_partials(tokens, code) == parts
    m = lambda rows: -(-rows // 128)
    steps = sorted({1, 2, tokens // 2, tokens} | {v for v in (127, 128, 129) if v <= tokens})
    for a in steps:
        for b in steps:
            for c in steps:
                d = 2 * tokens - a - b - c
                if 0 <= d <= tokens:
                    assert ((m(a) + m(b) + m(c) + m(d)) * parts + m(tokens) * shared) * 10 <= 256


def test_many_experts_keep_the_rule_by_the_mean_segment():
    assert few_rows_partials(64, _lib.W_E4M3FN, experts=16) == 1   # 17 tiles by 10: two parts are no round

#!/usr/bin/env python3
"""Writes swiglu224_asm.inc: the assembly of the fp8 gate/up kernel on 224-token tiles (swiglu224.h). Run by the build.

    python comfyui_amd/csrc/gen_swiglu224.py [output file]

One wave per SIMD (4 waves, 512 registers each) on a tile of 224 tokens x 256 weight rows (the same 128 features of w1 and w3),
wave tile 112 x 128 of v_mfma_f32_16x16x128_f8f6f4. A K step is 128 bytes, one MFMA deep, through two LDS stages; its 56 MFMAs go
in quadrants (weights 0-3 / 4-7 x token blocks 0-3 / 4-6), and the fragments of quadrants that are done are refilled from the
next stage. The epilogue of a tile packs w1 x and w3 x (scaled, rounded to bf16) into words: 28 pieces of 4 words per lane, 22 of
them stay in registers, 6 go to LDS. SiLU, product, cast and stores are issued behind the MFMAs of the next tile's first 7
pairs of K steps (a token block per pair; these pairs are written out, the others are a loop).

A low tile has 128 tokens, 4 blocks per wave: the same loads (slabs without rows ask for nothing) and 32 MFMAs a step, in two texts, behind a
tile of 7 and behind a low one.

Register map (per wave):
  a[0:223]    accumulators acc[ft][tt] = a[(7*ft + tt)*4 : +3], ft: 16 weight rows (0-3 w1, 4-7 w3), tt: 16 tokens
  a[224:255]  weight fragments 0-3 (8 registers each)
  v[128:159]  token fragments 0-3, v[160:183] token fragments 4-6, v[184:215] weight fragments 4-7; the last two are the
              epilogue's work registers
  v[38:85], v[216:255]  the deferred pieces
  v[88:94]    row indices of the tile after the next
  v[96:127]   addresses (CTX below) and work registers
  v[34:37]    finished outputs of a token block
  s[64:75]    buffer resources of the loads: tokens, w1, w3; s[76:78] weight offsets of a step
  v[0:33]     left to the compiler
"""
import os
import sys

HERE = os.path.dirname(os.path.abspath(__file__))
sys.path.insert(0, HERE)
from gen_gemm4w import DRAIN_WAIT, STAGE, W_TILE, Feeder, check_trans, quad  # noqa: E402

OUT = os.path.join(HERE, "swiglu224_asm.inc")
NTT = 7
LOW = 4                                           # 16-token blocks of a wave in a low tile
CTX = 96
TOK_ADDR = [CTX + 0, CTX + 1]                     # LDS address of the lane's token fragment, per 64-byte half of a step
W_ADDR = [CTX + 2, CTX + 3]
TOK_VOFF = [CTX + 4 + j for j in range(NTT)]      # global byte offset of the lane's row of token slab j
W_VOFF = CTX + 11                                 # same for weight slab 0; the others' distance goes in a scalar register
NEXT = [CTX + 12 + j for j in range(NTT)]         # TOK_VOFF of the next tile
DEF_ST = CTX + 19                                 # output byte offset of the lane in the deferred token block
GATHER_VOFF = CTX + 20                            # byte offset of the lane's entry of slabs 0-2 in the row index list, less 128 per slab
STG = CTX + 21                                    # LDS address of the lane's deferred pieces
GATHER_VOFF3, GATHER_VOFF4 = CTX + 22, CTX + 23   # of slab 3, which holds rows of both wave rows, and of slabs 4-6
TMP = CTX + 24                                    # v[120:126]
GATHER = 88
RES = 34
PIECES = [38 + 4 * i for i in range(12)] + [216 + 4 * i for i in range(10)]   # pieces 0-21 = token block * 4 + ft
IN_LDS = list(range(len(PIECES), 4 * NTT))        # the others; read back into the registers of the first ones


class At:
    """Positions (MFMA index within a step) of the events, by the tile's token blocks per wave."""
    def __init__(self, nt):
        self.m = 8 * nt
        self.free = 16              # the stage has been read; barrier
        self.load = [17 + round((2.55 if nt == NTT else 1) * j) for j in range(15)]
        self.land = {NTT: 38, LOW: 26}[nt]   # the next stage has landed; barrier, then the reads of the next step's first quadrant
        self.store = self.m - 1     # odd step: a finished token block
        self.stg = 8                # reads of deferred pieces from LDS


def weight(f):
    return f"a[{224 + 8 * f}:{231 + 8 * f}]" if f < 4 else f"v[{184 + 8 * (f - 4)}:{191 + 8 * (f - 4)}]"


def token(t):
    return f"v[{128 + 8 * t}:{135 + 8 * t}]"


def half(reg, h):
    c, lo = reg[0], int(reg[2:].split(":")[0])
    return f"{c}[{lo + 4 * h}:{lo + 4 * h + 3}]"


def reads(stage, frags):
    return [f"ds_read_b128 {half(weight(i) if k == 'w' else token(i), h)}, v{(W_ADDR if k == 'w' else TOK_ADDR)[h]} offset:{stage * STAGE + 2048 * i}"
            for k, i in frags for h in range(2)]


def blocks(stage, nt):
    """Token blocks of the first and of the second quadrant."""
    cut = (nt + 1) // 2
    return (range(0, cut), range(cut, nt)) if stage == 0 else (range(cut, nt), range(0, cut))


def first_reads(stage, nt):
    t = list(blocks(stage, nt)[0])
    return reads(stage, [("w", 0), ("t", t[0]), ("w", 1), ("w", 2), ("w", 3)] + [("t", x) for x in t[1:]])


def own_reads(stage, nt):
    return reads(stage, [("t", x) for x in blocks(stage, nt)[1]] + [("w", f) for f in range(4, 8)])


def mfma_order(stage, nt):
    t0, t1 = blocks(stage, nt)
    o = []
    for fts, tts in ((range(4), t0), (range(4), t1), (range(4, 8), t1), (range(4, 8), t0)):
        for k, tt in enumerate(tts):
            o += [(ft, tt) for ft in (fts if k % 2 == 0 else reversed(fts))]
    return o


def loads(stage):
    """(m0, load) of a step into `stage`: 7 slabs of 32 tokens, 8 of 32 weight rows. LDS rows of a wave's 128: ft 0-3 are 64 rows of w1, 4-7
    the same of w3; slab j starts at weight row (j >> 2) * 64 + (j & 1) * 8 (swiglu224.h)."""
    out = [(f"s_add_u32 m0, %[ldsw], {stage * STAGE + j * 4096}", f"buffer_load_dwordx4 v{TOK_VOFF[j]}, s[64:67], %[so] offen lds") for j in range(NTT)]
    for j in range(8):
        rs = "s[68:71]" if (j // 2) % 2 == 0 else "s[72:75]"
        so = ("%[so]", "s76", "s77", "s78")[(j >> 2) * 2 + (j & 1)]
        out.append((f"s_add_u32 m0, %[ldsw], {W_TILE + stage * STAGE + j * 4096}", f"buffer_load_dwordx4 v{W_VOFF}, {rs}, {so} offen lds"))
    return out


def silu_words(src, dst, clamp):
    """Four words (low half bf16(w1 x), high half bf16(w3 x)) src.. -> four e4m3fn bytes in dst: s = bf16(silu(g)), m = bf16(s u),
    e4m3fn(bf16(m %[inv])), or clamp: e4m3fn(m within +-%[inv]), NaN as it is; two values at a time: list of (instruction, cycles)."""
    ga, ua, gb, ub, ta, tb, pk = range(TMP, TMP + 7)
    o = []
    for p in range(2):
        da, db = src + 2 * p, src + 2 * p + 1
        o += [(f"v_lshlrev_b32 v{ga}, 16, v{da}", 4), (f"v_lshlrev_b32 v{gb}, 16, v{db}", 4),
              (f"v_mul_f32 v{ta}, 0xbfb8aa3b, v{ga}", 4), (f"v_mul_f32 v{tb}, 0xbfb8aa3b, v{gb}", 4),
              (f"v_exp_f32 v{ta}, v{ta}", 16), (f"v_exp_f32 v{tb}, v{tb}", 16),
              (f"v_and_b32 v{ua}, 0xffff0000, v{da}", 4), (f"v_and_b32 v{ub}, 0xffff0000, v{db}", 4),
              (f"v_add_f32 v{ta}, 1.0, v{ta}", 4), (f"v_add_f32 v{tb}, 1.0, v{tb}", 4),
              (f"v_rcp_f32 v{ta}, v{ta}", 16), (f"v_rcp_f32 v{tb}, v{tb}", 16), ("s_nop 0", 4),
              (f"v_mul_f32 v{ta}, v{ga}, v{ta}", 4), (f"v_mul_f32 v{tb}, v{gb}, v{tb}", 4),
              (f"v_cvt_pk_bf16_f32 v{pk}, v{ta}, v{tb}", 4),
              (f"v_lshlrev_b32 v{ta}, 16, v{pk}", 4), (f"v_and_b32 v{tb}, 0xffff0000, v{pk}", 4),
              (f"v_mul_f32 v{ta}, v{ta}, v{ua}", 4), (f"v_mul_f32 v{tb}, v{tb}, v{ub}", 4),
              (f"v_cvt_pk_bf16_f32 v{pk}, v{ta}, v{tb}", 4),
              (f"v_lshlrev_b32 v{ta}, 16, v{pk}", 4), (f"v_and_b32 v{tb}, 0xffff0000, v{pk}", 4),
              *([(f"v_minimum3_f32 v{t}, v{t}, %[inv], %[inv]", 4) for t in (ta, tb)] + [(f"v_maximum3_f32 v{t}, v{t}, -%[inv], -%[inv]", 4) for t in (ta, tb)]
                if clamp else [(f"v_mul_f32 v{t}, %[inv], v{t}", 4) for t in (ta, tb)]),
              (f"v_cvt_pk_bf16_f32 v{pk}, v{ta}, v{tb}", 4),
              (f"v_cvt_scalef32_pk_fp8_bf16 v{dst}, v{pk}, 1.0" + (" op_sel:[0,0,1]" if p else ""), 4)]
    return o


def piece_at(i):
    return PIECES[i] if i < len(PIECES) else PIECES[i - len(PIECES)]


def step(stage, first, block, stored, nt, clamp):
    """One K step out of `stage`. Entry: the reads of its first quadrant are in flight. first: the accumulators start from zero.
    block: the deferred token block of this pair of steps (two of its pieces per step), None = none. stored: the step before ended with a
    store for certain."""
    L = []
    at = At(nt)
    order, own, nxt = mfma_order(stage, nt), own_reads(stage, nt), first_reads(stage ^ 1, nt)
    events = dict(zip(at.load, loads(stage)))
    pieces = [] if block is None else [4 * block + 2 * stage, 4 * block + 2 * stage + 1]
    from_lds = [i for i in pieces if i in IN_LDS]
    start = at.free if from_lds else 0
    work = Feeder([op for i in pieces for op in silu_words(piece_at(i), RES + i % 4, clamp)], at.store - 2 - start)
    n_first = 4 * len(blocks(stage, nt)[0])
    L += ["s_add_u32 s76, %[so], %[kb8]", "s_add_u32 s77, %[so], %[kb64]", "s_add_u32 s78, s76, %[kb64]"]
    for q, (ft, tt) in enumerate(order):
        if q == 0:
            L.append("s_waitcnt lgkmcnt(0)")
        if q == n_first and q < at.free:   # the second quadrant's tokens are there, its weights are the first's
            L.append("s_waitcnt lgkmcnt(8)")
        if q in events:
            L.append(events[q][0])
        acc = f"a[{(NTT * ft + tt) * 4}:{(NTT * ft + tt) * 4 + 3}]"
        L.append(f"v_mfma_f32_16x16x128_f8f6f4 {acc}, {weight(ft)}, {token(tt)}, {'0' if first else acc}")
        if q in events:
            L.append(events[q][1])
        if q < 8:
            L += own[2 * q:2 * q + 2]
        if q == at.stg:
            L += [f"ds_read_b128 {quad(piece_at(i))}, v{STG} offset:{1024 * IN_LDS.index(i)}" for i in from_lds]
        if q == at.free - 1:
            L += ["s_waitcnt lgkmcnt(0)", "s_barrier"]
        if q == at.land - 1:
            # requests return in order: those of this step and the store are younger than the next step's operands
            L += [f"s_waitcnt vmcnt({sum(p < at.land for p in at.load) + stored})", "s_barrier"]
        if q >= at.land:
            L += nxt[2 * (q - at.land):2 * (q - at.land) + 2]
        if start <= q < at.store - 2:
            L += work.take()
        if q == at.store and block is not None and stage == 1:
            L += [f"buffer_store_dwordx4 {quad(RES)}, v{DEF_ST}, %[dro], 0 offen", f"v_add_u32 v{DEF_ST}, %[dldo], v{DEF_ST}"]
    assert work.done() and len(own) <= 16 and len(nxt) <= 2 * (len(order) - at.land)
    # a fragment is overwritten behind the last MFMA that reads it
    last = {}
    for q, (ft, tt) in enumerate(order):
        last[("w", ft)] = last[("t", tt)] = q
    for k, r in enumerate(nxt):
        for key, reg in [(("w", f), weight(f)) for f in range(8)] + [(("t", t), token(t)) for t in range(nt)]:
            if any(half(reg, h) in r for h in range(2)):
                assert last[key] <= at.land + k // 2, (stage, key)
    L.append("s_add_u32 %[so], %[so], 128")
    return L


def pair(first, block, nt, clamp):
    return step(0, first, block, block not in (None, 0), nt, clamp) + step(1, False, block, False, nt, clamp)


def k_loop(nt, before, clamp):
    """All K steps of a tile of nt blocks in pairs, %[n] of them (at least 8), behind a tile of `before`. Before the last pair the loads turn
    to the first two steps of the next tile and the row indices of the tile after it are requested. The last step reads the first quadrant of
    the next tile's first one: a lower tile's is part of it."""
    L = ["s_mov_b64 s[64:65], %[ra]", "s_mov_b64 s[66:67], %[rah]", "s_mov_b64 s[68:69], %[rb]", "s_mov_b64 s[70:71], %[rbh]",
         "s_mov_b64 s[72:73], %[rc]", "s_mov_b64 s[74:75], %[rbh]", f"s_sub_u32 %[n], %[n], {before}"]
    for b in range(before):
        L += pair(b == 0, b, nt, clamp)
    L += ["11:", "s_cmp_eq_u32 %[n], 1", "s_cbranch_scc1 13f", "14:"] + pair(False, None, nt, clamp)
    L += ["s_sub_u32 %[n], %[n], 1", "s_cmp_lg_u32 %[n], 0", "s_cbranch_scc1 11b", "s_branch 12f"]
    L += ["13:", "s_mov_b64 s[64:65], %[na]", "s_mov_b64 s[66:67], %[nah]", "s_mov_b64 s[68:69], %[nb]", "s_mov_b64 s[72:73], %[nc]",
          "s_mov_b32 s70, %[nbn]", "s_mov_b32 s74, %[nbn]", "s_mov_b32 %[so], 0"]
    L += [f"v_mov_b32 v{TOK_VOFF[j]}, v{NEXT[j]}" for j in range(NTT)]
    for j in range(NTT):
        v, off = (GATHER_VOFF, 128 * j) if j < 3 else (GATHER_VOFF3, 0) if j == 3 else (GATHER_VOFF4, 128 * (j - 4))
        L.append(f"buffer_load_dword v{GATHER + j}, v{v}, %[gr], 0 offen offset:{off}")
    return L + ["s_branch 14b", "12:", "s_nop 15"]


def epilogue(nt):
    """acc * scale rounded to bf16, w1 x and w3 x packed into a word; work registers v[160:215]."""
    L = []
    for i in range(4 * nt):
        tt, ft = divmod(i, 4)
        w = 160 + 12 * (i % 4)
        for e in range(4):
            L += [f"v_accvgpr_read_b32 v{w + 2 * e}, a{(NTT * ft + tt) * 4 + e}",
                  f"v_accvgpr_read_b32 v{w + 2 * e + 1}, a{(NTT * (ft + 4) + tt) * 4 + e}"]
        for e in range(4):
            L += [f"v_mul_f32 v{w + 2 * e}, %[sc], v{w + 2 * e}", f"v_mul_f32 v{w + 2 * e + 1}, %[su], v{w + 2 * e + 1}"]
        dst = w + 8 if i in IN_LDS else PIECES[i]
        for e in range(4):
            L.append(f"v_cvt_pk_bf16_f32 v{dst + e}, v{w + 2 * e}, v{w + 2 * e + 1}")
        if i in IN_LDS:
            L.append(f"ds_write_b128 v{STG}, {quad(dst)} offset:{1024 * IN_LDS.index(i)}")
    return L


def tile(clamp):
    """A tile by its text, %[text]: 0 = 7 blocks behind a tile of 7, 1 = a low one behind a tile of 7, 2 = a low one behind a low one. (The
    blocks' tiles go from high to low.)"""
    L = ["s_cmp_eq_u32 %[text], 1", "s_cbranch_scc1 101f", "s_cmp_eq_u32 %[text], 2", "s_cbranch_scc1 102f"]
    L += k_loop(NTT, NTT, clamp) + epilogue(NTT) + ["s_branch 109f", "101:"] + k_loop(LOW, NTT, clamp) + epilogue(LOW)
    return L + ["s_branch 109f", "102:"] + k_loop(LOW, LOW, clamp) + epilogue(LOW) + ["109:"]


def drain(clamp):
    """The deferred pieces of a block's last tile, with nothing to hide behind; %[text] other than 0: a low one."""
    L = []
    for tt in range(NTT):
        if tt == LOW:
            L += ["s_cmp_lg_u32 %[text], 0", "s_cbranch_scc1 21f"]
        for g in range(4):
            i = 4 * tt + g
            if i in IN_LDS:
                L += [f"ds_read_b128 {quad(piece_at(i))}, v{STG} offset:{1024 * IN_LDS.index(i)}", "s_waitcnt lgkmcnt(0)"]
            L += [op for op, _ in silu_words(piece_at(i), RES + g, clamp)]
        L += [f"buffer_store_dwordx4 {quad(RES)}, v{DEF_ST}, %[dro], 0 offen", f"v_add_u32 v{DEF_ST}, %[dldo], v{DEF_ST}"]
    return L + ["21:", "s_nop 7"]


def generate():
    out = ["// Generated by gen_swiglu224.py; do not edit. See that script for the register map and the schedule.", ""]
    for name, lines in (("HDMOE_S224_TILE", tile(False)), ("HDMOE_S224_FILL", first_reads(0, NTT)), ("HDMOE_S224_DRAIN", DRAIN_WAIT + drain(False)),
                        ("HDMOE_S224_TILE_CLAMP", tile(True)), ("HDMOE_S224_DRAIN_CLAMP", DRAIN_WAIT + drain(True))):
        check_trans(lines)
        out.append(f"#define {name} \\")
        out.append(" \\\n".join('  "' + ln + '\\n"' for ln in lines))
        out.append("")
    return "\n".join(out)


if __name__ == "__main__":
    path = sys.argv[1] if len(sys.argv) > 1 else OUT
    text = generate()
    if not os.path.exists(path) or open(path).read() != text:
        with open(path, "w") as f:
            f.write(text)

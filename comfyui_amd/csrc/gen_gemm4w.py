#!/usr/bin/env python3
"""Writes gemm4w_asm.inc: the assembly of the 4-wave GEMM (gemm4w.h). Run by the build.

    python comfyui_amd/csrc/gen_gemm4w.py [output file]

One wave per SIMD (4 waves, 512 registers each) on a 256-token x 256-weight-row tile, wave tile 128 x 128 of
v_mfma_f32_16x16x32. Token block tt of wave pair wt is rows 32 tt + 16 wt of the tile, so a tile with fewer tokens is one with fewer
token blocks: with 16-bit activations there is a text for each of HEIGHTS, and a tile runs the one of its size. A pair of K steps
that ends a tile of fewer blocks still fetches all of the next tile, whatever its height. A K step is 64 elements (128 bytes per token row) through two LDS stages. The fragments of both
32-element slices of a step have registers of their own, so a stage has been read for good after about a third of its
step, and the global->LDS loads of the step after the next go into it from there on: they have about 1.4 steps to
arrive. Two barriers per step: everyone has read this stage; everyone's loads of the next one have landed. One statement
holds the K loop and the epilogue of a tile, so that no accumulator crosses compiled code.

Weights of one byte (w8: e4m3fn) are loaded by the pair of K steps (128 bytes per row), read 8 bytes per lane and
converted to bf16 on the way to the matrix cores (exact), 64 conversions beside the 128 MFMAs of a step.

fp8 (F8: e4m3fn activations and weights): a K step of 128 elements is one v_mfma_f32_16x16x128_f8f6f4 deep. See step8.

GELU: an epilogue leaves the rounded sums of a tile in a scratch buffer of the block's own (it stays in the caches); while
the next tile multiplies, the wave reads them back 16 bytes per lane at a time, applies the activation and stores the
outputs, one piece per K step behind the MFMAs.

Register map (per wave):
  a[0:255]    accumulators acc[ft][tt] = a[(8*ft + tt)*4 : +3], ft: 16 weight rows, tt: 16 tokens
  v[128:159]  token fragments of slice 0, v[160:191] weight fragments of slice 0 (4 registers each, tt / ft ascending)
  v[192:223]  token fragments of slice 1, v[224:255] weight fragments of slice 1; work registers of the epilogue
              (F8: tt / ft 0-3 in v[128:159] / v[160:191], 4-7 in v[192:223] / v[224:255], 8 registers each)
  v[96:127]   addresses (CTX below)
  v[80:95]    row offsets of the next tile, v[72:79] row indices of the tile after the next
  v[34:71]    work registers of the K loop
  s[64:75]    buffer resources of the loads: tokens, weights (rows 0-63 and 64-127 of either half)
  v[0:33]     left to the compiler
"""
import os
import sys

HERE = os.path.dirname(os.path.abspath(__file__))
OUT = os.path.join(HERE, "gemm4w_asm.inc")

CTX = 96
TOK_ADDR = [CTX + 0, CTX + 1]                     # LDS address of the lane's token fragment, per slice
W_ADDR = [CTX + 2, CTX + 3]                       # same for weights; w8: per slice of the even step (the odd one flips bit 6)
TOK_VOFF = [CTX + 4 + j for j in range(8)]        # global byte offset of the lane's row of token slab j
W_VOFF = [CTX + 12 + j for j in range(8)]         # same for weight slab j
OUT_VOFF = CTX + 20                               # output byte offset of the lane: its token, its 8 features of group 0
ROW_VOFF = CTX + 21                               # running copy of it
GATHER_VOFF = CTX + 22                            # byte offset of the lane's entry of slab 0 in the row index list
BIAS_VOFF = CTX + 23                              # byte offset of the lane's first bias of the tile
DEF_LD, DEF_ST = CTX + 24, CTX + 25               # GELU: offset in the scratch of the piece read back, in the output of the one stored
SCR_VOFF = CTX + 26                               # GELU: the lane's offset in the scratch
NEXT = 80                                         # v[80:95]: TOK_VOFF and W_VOFF of the next tile
GATHER = 72                                       # v[72:79]
BIAS = 56                                         # v[56:71]: 8 quads of 16-bit biases
PIECE = [34, 38]                                  # GELU: pieces read back, by step parity
RES = 42                                          # GELU: finished piece
TMP = 46                                          # GELU: v[46:55]
RAW = 40                                          # w8: v[40:55] weight bytes of a slice, 2 registers per ft
STAGE = 32768                                     # bytes of one stage of the token tile = of the weight tile
W_TILE = 65536                                    # LDS: [tok 0 | tok 1 | w 0 | w 1]
FRAG = {("a", 0): 128, ("b", 0): 160, ("a", 1): 192, ("b", 1): 224}
MFMA = {"BF16": "v_mfma_f32_16x16x32_bf16", "F16": "v_mfma_f32_16x16x32_f16"}
PK = {"BF16": "v_cvt_pk_bf16_f32", "F16": "v_cvt_pk_f16_f32", "F8": "v_cvt_pk_bf16_f32"}   # F8: the outputs are bf16

HEIGHTS = (8, 7, 6, 5, 4)                         # token blocks of a wave: 32 tokens of the tile each


class At:
    """Positions (MFMA index within a slice of `m`) of the events of a step of `nt` token blocks. last: of the pair that ends a
    tile, which fetches 8 token blocks whatever nt is."""
    def __init__(self, nt, last=False):
        self.nt, self.m, self.last = nt, 8 * nt, last
        self.loads = 8 if last else nt          # token loads of a step
        self.free = 16 + nt                     # slice 0: the stage has been read (8 + nt reads, one per MFMA); barrier
        self.load = self.free + 1               # first load of the step after the next, and MFMAs between two loads
        self.every = (2 * self.m - self.load - 8) // (self.loads + 7)
        self.land = self.m - 16 - 2 * nt        # slice 1: the next stage has landed; barrier, then the reads of slice 0 of the next step
        self.cvt1 = self.free + 2               # w8, slice 0: first conversion of slice 1
        self.st, self.ld = self.m - 7, self.m - 4   # GELU, slice 0: piece stored, piece read back


class At8:
    """The same for an fp8 step of `nt` token blocks, 8 nt MFMAs in quadrants: weights 0-3 / 4-7 by the token blocks `halves`."""
    def __init__(self, nt, stage, last=False):
        self.m = 8 * nt
        h = (nt + 1) // 2
        self.halves = (range(h), range(h, nt)) if stage == 0 else (range(h, nt), range(h))
        first, second = (len(t) for t in self.halves)
        self.loads = 8 if last else nt
        self.free = 4 * first                       # the stage has been read; barrier
        self.land = 4 * first + 8 * second - 4      # the next stage has landed; barrier, then the reads of the next step's first quadrant
        n, lo = self.loads + 8, self.free + 2
        self.load_at = [lo + 3 * j if nt == 8 else lo + j * (self.m - lo) // n for j in range(n)]
        assert self.load_at[-1] < self.m and len(set(self.load_at)) == n


def quad(b):
    return f"v[{b}:{b + 3}]"


def reads(stage, ks, w8, odd, nt=8):
    """The 8 + nt fragment reads of a slice, in the order the MFMAs want them."""
    order = [("b", 0)] + [("a", t) for t in range(nt)] + [("b", f) for f in range(1, 8)]
    if w8:
        order.sort(key=lambda o: o[0] == "a")     # the weights have to be converted
    out = []
    for kind, i in order:
        if kind == "b" and w8:
            # 16 rows of 128 bytes per ft; odd steps read the upper 64 bytes of a row (the swizzle is an xor, so the
            # address of the upper half is the lower one's with bit 6 flipped: a second address register)
            out.append(f"ds_read_b64 v[{RAW + 2 * i}:{RAW + 2 * i + 1}], v{W_ADDR[ks]} offset:{2048 * i}")
        else:
            out.append(f"ds_read_b128 {quad(FRAG[(kind, ks)] + 4 * i)}, v{(TOK_ADDR if kind == 'a' else W_ADDR)[ks]} "
                       f"offset:{stage * STAGE + (4096 if kind == 'a' else 2048) * i}")
    return out


def token_loads(stage, nt=8):
    return [(f"s_add_u32 m0, %[ldsw], {stage * STAGE + j * 4096}",
             f"buffer_load_dwordx4 v{TOK_VOFF[j]}, s[64:67], %[so] offen lds") for j in range(nt)]


def weight_loads(stage, w8):
    out = []
    for j in range(8):
        rs = "s[68:71]" if (j // 2) % 2 == 0 else "s[72:75]"
        m0 = f"s_add_u32 m0, %[ldswb], {j * 4096}" if w8 else f"s_add_u32 m0, %[ldsw], {W_TILE + stage * STAGE + j * 4096}"
        out.append((m0, f"buffer_load_dwordx4 v{W_VOFF[j]}, {rs}, {'%[wso]' if w8 else '%[so]'} offen lds"))
    return out


def mfma_order(nt):
    o = []
    for ft in range(8):
        o += [(ft, tt) for tt in (range(nt) if ft % 2 == 0 else range(nt - 1, -1, -1))]
    return o


def unpack(dt, dst, src, hi):
    if dt in ("BF16", "F8"):
        return f"v_and_b32 v{dst}, 0xffff0000, {src}" if hi else f"v_lshlrev_b32 v{dst}, 16, {src}"
    return f"v_cvt_f32_f16_sdwa v{dst}, {src} dst_sel:DWORD dst_unused:UNUSED_PAD src0_sel:WORD_{int(hi)}"


# Q(a) = 1 - Phi(a) = exp(-a^2 / 2) * P(t), t = 1 / (1 + 0.3 a): coefficients of t^1 .. t^8, fitted here to
# erfcx(a / sqrt 2) / 2 on [0, 14] (relative error 1.5e-7, 7e-7 when evaluated in fp32)
GELU_P = 0.3        # gemm4w.h passes gk and gp = 0.3 / gk
GELU_C = [0.1196293, 0.12075395, 0.09991351, 0.12856157, -0.05368355, 0.2063534, -0.15720303, 0.03567476]


def f32(v):
    import struct
    return "0x%08x" % struct.unpack("<I", struct.pack("<f", v))[0]


def gelu_words(dt, src, dst, n):
    """gelu(x) = (x + |x|) / 2 - |x| Q(|x|) of n packed words src.. -> dst.., two values at a time in the work registers
    TMP..TMP+9: list of (instruction, cycles). No cancellation, so the negative tail keeps its digits; infinities and NaN
    come out as 0.5 x (1 + erf) has them (the legacy product takes 0 * inf as 0). |x| is carried as a = k |x|,
    k^2 = log2(e) / 2, so that exp(-x^2 / 2) is one square and one exp2; the factor is folded into the other constants. bf16:
    x is halved first, x + |x| would overflow above 1.7e38 (%[gk] is 2 k there)."""
    k = (0.5 * 1.4426950408889634) ** 0.5
    c = [v / k for v in GELU_C]
    o = []
    for w in range(n):
        x, a, d, e, p = ((TMP + i, TMP + 5 + i) for i in range(5))

        def both(f, cyc=4):
            o.extend((f(i), cyc) for i in range(2))
        both(lambda i: unpack(dt, x[i], f"v{src + w}", i == 1))
        if dt == "BF16":
            both(lambda i: f"v_mul_f32 v{x[i]}, 0.5, v{x[i]}")
        both(lambda i: f"v_mul_f32 v{a[i]}, |v{x[i]}|, %[gk]")
        both(lambda i: f"v_fma_f32 v{d[i]}, v{a[i]}, %[gp], 1.0")
        both(lambda i: f"v_rcp_f32 v{d[i]}, v{d[i]}", 16)
        both(lambda i: f"v_mul_f32 v{e[i]}, v{a[i]}, v{a[i]}")
        both(lambda i: f"v_exp_f32 v{e[i]}, -v{e[i]}", 16)
        both(lambda i: f"v_mul_f32 v{p[i]}, {f32(c[7])}, v{d[i]}")
        both(lambda i: f"v_add_f32 v{p[i]}, {f32(c[6])}, v{p[i]}")
        for v in reversed(c[:6]):
            both(lambda i: f"v_fmaak_f32 v{p[i]}, v{p[i]}, v{d[i]}, {f32(v)}")
        both(lambda i: f"v_mul_f32 v{p[i]}, v{p[i]}, v{d[i]}")
        both(lambda i: f"v_mul_f32 v{p[i]}, v{p[i]}, v{e[i]}")
        both(lambda i: f"v_mul_legacy_f32 v{p[i]}, v{p[i]}, v{a[i]}")
        both(lambda i: f"v_add_f32 v{x[i]}, v{x[i]}, |v{x[i]}|")
        both(lambda i: f"v_sub_f32 v{x[i]}, v{x[i]}, v{p[i]}" if dt == "BF16" else f"v_fma_f32 v{x[i]}, v{x[i]}, 0.5, -v{p[i]}")
        o.append((f"{PK[dt]} v{dst + w}, v{x[0]}, v{x[1]}", 4))
    return o


# a resource that the compiler has just read back from a vector register's lanes may not be used by a load before 5 wait states
DRAIN_WAIT = ["s_nop 4"]


class Feeder:
    """Hands instructions out evenly over a number of places."""
    def __init__(self, ops, places):
        self.ops, self.pos, self.spent, self.given = ops, 0, 0, 0.0
        self.share = sum(c for _, c in ops) / max(1, places)

    def take(self):
        out = []
        self.given += self.share
        while self.pos < len(self.ops) and self.spent < self.given - 1e-9:
            out.append(self.ops[self.pos][0])
            self.spent += self.ops[self.pos][1]
            self.pos += 1
        return out

    def done(self):
        return self.pos == len(self.ops)


def conversions(ks):
    """w8: the slice's weight bytes to bf16, in the order of the reads."""
    o = []
    for ft in range(8):
        for h in range(4):
            o.append((f"v_cvt_scalef32_pk_bf16_fp8 v{FRAG[('b', ks)] + 4 * ft + h}, v{RAW + 2 * ft + h // 2}, 1.0"
                      + (" op_sel:[1,0,0]" if h % 2 else ""), 4))
    return o


def requests(w8, gelu, stage, at, first=False):
    """The vector-memory requests of a step out of `stage` (first: of a tile's first pair) as (position, kind), position =
    MFMA index over both slices."""
    n = at.loads + (0 if w8 and stage == 0 else 8)
    out = [(at.load + j * at.every, "t" if j < at.loads else "w") for j in range(n)]
    if gelu:
        out += ([] if first else [(at.st, "s")]) + [(at.ld, "l")]
    return sorted(out)


def young(w8, gelu, stage, at, first):
    """How many vector-memory requests may still be out when the next step's operands must have landed (requests return in
    order): those issued after the last one that is needed. Needed: the tokens (16-bit weights too) requested a step ago and
    the piece read back then; one-byte weights were requested two steps ago or earlier. The step before may be one of another
    height: what it issues behind the last needed request is the same for all."""
    before = [k for p, k in requests(w8, gelu, stage, at, first) if p < at.m + at.land]
    need = {"t", "l"} | (set() if w8 else {"w"})
    behind = set()
    for other in [At(nt, end) for nt in HEIGHTS for end in (False, True)]:
        after = 0
        for _, k in reversed(requests(w8, gelu, stage ^ 1, other)):
            if k in need:
                break
            after += 1
        behind.add(after)
    assert len(behind) == 1
    return behind.pop() + len(before)


def step(dt, w8, gelu, stage, first, at):
    """One K step out of `stage`. Entry: the reads of its slice 0 are in flight (lgkmcnt; w8: converted). first: of
    a tile's first pair, whose step 0 starts the accumulators from zero and which has no finished piece to store."""
    L = []
    order = mfma_order(at.nt)
    # w8: the even step's slice 1 and the odd step's slice 0 read the same weight stage; the next even step's slice 0 reads
    # the other one (W_ADDR is flipped between the pairs)
    rd1 = reads(stage, 1, w8, stage, at.nt)
    rd0 = reads(stage ^ 1, 0, w8, stage ^ 1, at.loads if stage == 1 else at.nt)
    ld = token_loads(stage, at.loads) + ([] if w8 and stage == 0 else weight_loads(stage, w8))
    # w8: first conversion of the next step's slice 0, when a few of the reads behind the 8 of the weights have been issued
    cvt0_at = at.land + 14 - (8 - at.nt) // 2
    cvt1, cvt0 = Feeder(conversions(1) if w8 else [], at.m - at.cvt1), Feeder(conversions(0) if w8 else [], at.m - cvt0_at)
    # the piece read back a step ago, in two parts around the end of the step (words n_b.. of the one before that first)
    n_b = 2
    half_b = Feeder(gelu_words(dt, PIECE[stage ^ 1], RES, n_b) if gelu else [], at.m - at.land)
    half_a = Feeder(gelu_words(dt, PIECE[stage] + n_b, RES + n_b, 4 - n_b) if gelu else [], at.st)
    assert len(rd1) <= at.free <= at.load and at.load + (at.loads + 7) * at.every < 2 * at.m and at.land + len(rd0) <= at.m
    for q in range(2 * at.m):
        ks, i = divmod(q, at.m)
        ft, tt = order[i]
        if q == 0:
            L.append("s_waitcnt lgkmcnt(0)")
        k = q - at.load
        now = ld[k // at.every] if k >= 0 and k % at.every == 0 and k // at.every < len(ld) else None
        if now:
            L.append(now[0])
        acc = f"a[{(8 * ft + tt) * 4}:{(8 * ft + tt) * 4 + 3}]"
        c = "0" if first and stage == 0 and ks == 0 else acc
        L.append(f"{MFMA[dt]} {acc}, {quad(FRAG[('b', ks)] + 4 * ft)}, {quad(FRAG[('a', ks)] + 4 * tt)}, {c}")
        if now:
            L.append(now[1])
        if ks == 0:
            if i < len(rd1):
                L.append(rd1[i])
            if i == at.free - 1:
                L += ["s_waitcnt lgkmcnt(0)", "s_barrier"]
            if w8 and i >= at.cvt1:
                L += cvt1.take()
            if gelu and i < at.st:
                L += half_a.take()
            if gelu and i == at.st:
                assert half_a.done()
            if gelu and i == at.st and not first:
                L.append(f"buffer_store_dwordx4 {quad(RES)}, v{DEF_ST}, %[dro], 0 offen offset:{64 * stage}")
            if gelu and i == at.ld:
                L.append(f"buffer_load_dwordx4 {quad(PIECE[stage])}, v{DEF_LD}, %[scr], 0 offen offset:{1024 * stage}")
        else:
            if i == at.land - 1:
                L += [f"s_waitcnt vmcnt({young(w8, gelu, stage, at, first)})", "s_barrier"]
                if w8 and stage == 1:   # the next pair's weights
                    L += [f"v_xor_b32 v{r}, {hex(STAGE)}, v{r}" for r in W_ADDR]
                if w8:                  # the other 64 bytes of the rows
                    L += [f"v_xor_b32 v{r}, 64, v{r}" for r in W_ADDR]
            if 0 <= i - at.land < len(rd0):
                L.append(rd0[i - at.land])
            if w8 and i == cvt0_at - 1:   # the weight bytes are there, the tokens may still be under way
                issued = min(len(rd0), cvt0_at - at.land)
                assert issued > 8
                L.append(f"s_waitcnt lgkmcnt({issued - 8})")
            if w8 and i >= cvt0_at:
                L += cvt0.take()
            if gelu and i >= at.land:
                L += half_b.take()
    assert half_b.done() and cvt0.done() and cvt1.done()
    L.append("s_add_u32 %[so], %[so], 128")
    return L


def frag8(kind, i):
    """fp8: the 8 registers of a fragment (32 bytes per lane: the places g and 4 + g of its row in LDS, g = lane / 16; f8_chunk in gemm4w.h)."""
    return FRAG[(kind, i // 4)] + 8 * (i % 4)


def reads8(stage, frags):
    out = []
    for kind, i in frags:
        for h in range(2):
            out.append(f"ds_read_b128 {quad(frag8(kind, i) + 4 * h)}, v{(TOK_ADDR if kind == 'a' else W_ADDR)[h]} "
                       f"offset:{stage * STAGE + (4096 if kind == 'a' else 2048) * i}")
    return out


def burst8(stage, nt=8):
    """The reads that a step out of `stage` starts from, and those it issues itself for its second half."""
    t0, t1 = ([("a", t) for t in h] for h in At8(nt, stage).halves)
    w0, w1 = [("b", f) for f in range(4)], [("b", f) for f in range(4, 8)]
    return reads8(stage, [w0[0], t0[0]] + w0[1:] + t0[1:]), reads8(stage, [t1[0], w1[0]] + t1[1:] + w1[1:])


def mfma_order8(nt, stage):
    """Four quadrants of MFMA tiles: (w0, t0), (w0, t1), (w1, t1), (w1, t0), t0 and t1 by step parity; token blocks outermost."""
    t0, t1 = At8(nt, stage).halves
    o = []
    for fts, tts in ((range(4), t0), (range(4), t1), (range(4, 8), t1), (range(4, 8), t0)):
        for k, tt in enumerate(tts):
            o += [(ft, tt) for ft in (fts if k % 2 == 0 else reversed(fts))]
    return o


def step8(stage, first, nt, last):
    """One fp8 K step out of `stage`: 128 bytes are one MFMA deep, so a step has no second slice to read ahead; its 8 nt MFMAs go in
    quadrants instead, and the fragments of quadrants that are done are refilled from the next stage. Entry: the reads of
    the first quadrant are in flight (burst8; of a tile's first step always those of 4 token blocks, whatever its height). last: of the pair
    that ends a tile."""
    L = []
    at = At8(nt, stage, last)
    order = mfma_order8(nt, stage)
    used = {}                                   # the last MFMA that reads a fragment
    for q, (ft, tt) in enumerate(order):
        used[("b", ft)] = used[("a", tt)] = q
    own = burst8(stage, nt)[1]
    nxt = burst8(stage ^ 1, nt)[0]
    ends = last and stage == 1
    if ends:                                    # token blocks 0-3, those that the last quadrant uses behind their last use
        nxt = burst8(0)[0]
    todo = [nxt[i:i + 2] for i in range(0, len(nxt), 2)]
    reg = {quad(frag8(k, i)): (k, i) for k in "ab" for i in range(8)}
    ld = token_loads(stage, at.loads) + weight_loads(stage, False)
    events = dict(zip(at.load_at, ld))
    assert len(own) // 2 <= at.free
    for q in range(at.m):
        ft, tt = order[q]
        if q == 0:
            L.append("s_waitcnt lgkmcnt(0)")
        now = events.get(q)
        if now:
            L.append(now[0])
        acc = f"a[{(8 * ft + tt) * 4}:{(8 * ft + tt) * 4 + 3}]"
        b, a = frag8("b", ft), frag8("a", tt)
        L.append(f"v_mfma_f32_16x16x128_f8f6f4 {acc}, v[{b}:{b + 7}], v[{a}:{a + 7}], {'0' if first and stage == 0 else acc}")
        if now:
            L.append(now[1])
        if q < 8:
            L += own[2 * q:2 * q + 2]
        if q == at.free - 1:
            L += ["s_waitcnt lgkmcnt(0)", "s_barrier"]
        if q == at.land - 1:   # the requests that may still be out are those of this step
            L += [f"s_waitcnt vmcnt({sum(p < at.land for p in at.load_at)})", "s_barrier"]
        # they overwrite fragments of the quadrants behind; those of the third are freed four MFMAs apart
        if q >= at.land and todo and used.get(reg[todo[0][0].split(" ", 1)[1].split(",")[0]], -1) <= q:
            L += todo.pop(0)
    assert not todo
    L.append("s_add_u32 %[so], %[so], 128")
    return L


def pair(dt, w8, gelu, first, at):
    if dt == "F8":
        return step8(0, first, at.nt, at.last) + step8(1, first, at.nt, at.last)
    L = []
    if gelu and not first:
        # pieces 2p, 2p + 1: the pair of K steps p (0..13) reads them back, pair p + 1 stores them (64 bytes per token each)
        L += [f"v_add_u32 v{DEF_LD}, 0x800, v{DEF_LD}", f"v_add_u32 v{DEF_ST}, %[dd], v{DEF_ST}", "s_sub_u32 %[dd], %[dldo], %[dd]",
              "s_sub_u32 %[dn], %[dn], 1", "s_cmp_ge_i32 %[dn], 0", "s_cbranch_scc1 21f", f"v_mov_b32 v{DEF_ST}, 0x80000000", "21:"]
    L += step(dt, w8, gelu, 0, first, at) + step(dt, w8, gelu, 1, first, at)
    if w8:   # the weight stage of the pair after the next is this pair's
        L += [f"s_xor_b32 %[ldswb], %[ldswb], {hex(STAGE)}", "s_add_u32 %[wso], %[wso], 128"]
    return L


def k_loop(dt, w8, gelu, bias, nt=8):
    """All K steps of a tile in pairs, %[n] of them (at least 2, w8: 3). Before the last pair the loads turn to the first
    two steps of the next tile; the row indices of the tile after it and this tile's biases are requested there too. w8:
    the weights of a pair are requested two pairs ahead, so they turn a pair earlier. The wait states at the end cover
    the distance between the last MFMA and the first read of an accumulator."""
    at, end = At(nt), At(nt, True)
    L = [f"s_mov_b64 s[{64 + 2 * i}:{65 + 2 * i}], %[r{i}]" for i in range(6)]
    L += pair(dt, w8, gelu, True, at) + ["s_sub_u32 %[n], %[n], 1", "11:"]
    wswitch = [f"s_mov_b64 s[{64 + 2 * i}:{65 + 2 * i}], %[nr{i}]" for i in range(2, 6)]
    wswitch += [f"v_mov_b32 v{W_VOFF[j]}, v{NEXT + 8 + j}" for j in range(8)]
    if w8:
        L += ["s_cmp_eq_u32 %[n], 2", "s_cbranch_scc1 15f", "16:"]
    L += ["s_cmp_eq_u32 %[n], 1", "s_cbranch_scc1 13f", "14:"]
    L += pair(dt, w8, gelu, False, at)
    L += ["s_sub_u32 %[n], %[n], 1", "s_cmp_lg_u32 %[n], 0", "s_cbranch_scc1 11b", "s_branch 12f"]
    if w8:
        L += ["15:"] + wswitch + ["s_mov_b32 %[wso], %[nwso]", "s_branch 16b"]
    L += ["13:", "s_mov_b64 s[64:65], %[nr0]", "s_mov_b64 s[66:67], %[nr1]", "s_mov_b32 %[so], %[nso]"]
    L += [f"v_mov_b32 v{TOK_VOFF[j]}, v{NEXT + j}" for j in range(8)]
    if not w8:
        L += wswitch
    L += [f"buffer_load_dword v{GATHER + j}, v{GATHER_VOFF}, %[gr], 0 offen offset:{128 * j}" for j in range(8)]
    if bias:
        L += [f"buffer_load_dwordx2 v[{BIAS + 2 * ft}:{BIAS + 2 * ft + 1}], v{BIAS_VOFF}, %[br], 0 offen "
              f"offset:{(ft >> 1) * 64 + (ft & 1) * 8}" for ft in range(8)]
    L += ["s_branch 14b"] if nt == 8 else pair(dt, w8, gelu, False, end)
    L += ["12:", "s_nop 15"]
    if gelu:   # the last piece read back is there: its registers are the compiler's between two tiles
        L.append(f"s_waitcnt vmcnt({sum(p > end.ld for p, _ in requests(False, True, 1, end))})")
    return L


def out_row(tt):
    return [f"v_add_u32 v{ROW_VOFF}, %[ldo32], v{ROW_VOFF}"] if tt else [f"v_mov_b32 v{ROW_VOFF}, v{OUT_VOFF}"]


def epilogue(dt, w8, bias, gelu, nt=8):
    """acc (* scale) (+ bias) rounded to 16 bits, 8 consecutive features (16 bytes) per lane and store, 64 bytes per token.
    v[192:223]: the lane's 32 biases, v[224:255] work. gelu: the first token block is activated at once, the others are
    left to the next tile's K loop."""
    L = []
    if bias:
        for ft in range(8):
            for h in range(4):
                L.append(unpack(dt, 192 + ft * 4 + h, f"v{BIAS + 2 * ft + h // 2}", h % 2))
    n = 0
    if gelu:
        L.append(f"v_mov_b32 v{DEF_LD}, v{SCR_VOFF}")
    for tt in range(nt):
        L += out_row(tt) if not (gelu and tt) else []
        for g in range(4):
            w = 224 + 16 * (n % 2)          # 8 values, then 4 packed words
            o = w + 8
            n += 1
            for p in range(2):
                for e in range(4):
                    L.append(f"v_accvgpr_read_b32 v{w + p * 4 + e}, a{(8 * (2 * g + p) + tt) * 4 + e}")
            for p in range(2):
                for e in range(4):
                    v, b = w + p * 4 + e, 192 + (2 * g + p) * 4 + e
                    if dt == "F8" and bias:   # the product is rounded before the bias is added, as the 8-wave kernel has it
                        L += [f"v_mul_f32 v{v}, %[sc], v{v}", f"v_add_f32 v{v}, v{b}, v{v}"]
                    elif w8 and bias:
                        L.append(f"v_fma_f32 v{v}, v{v}, %[sc], v{b}")
                    elif w8 or dt == "F8":
                        L.append(f"v_mul_f32 v{v}, %[sc], v{v}")
                    elif bias:
                        L.append(f"v_add_f32 v{v}, v{b}, v{v}")
            for q in range(4):
                L.append(f"{PK[dt]} v{o + q}, v{w + 2 * q}, v{w + 2 * q + 1}")
            if gelu and tt == 0:
                L += [i for i, _ in gelu_words(dt, o, o, 4)]
            if gelu and tt:
                L.append(f"buffer_store_dwordx4 {quad(o)}, v{DEF_LD}, %[scr], 0 offen offset:{1024 * g}")
            else:
                L.append(f"buffer_store_dwordx4 {quad(o)}, v{ROW_VOFF}, %[ro], 0 offen offset:{64 * g}")
        if gelu and tt in range(1, nt - 1):
            L.append(f"v_add_u32 v{DEF_LD}, 0x1000, v{DEF_LD}")
    return L


def swiglu_epilogue(w8, nt=8):
    """bf16(bf16(silu(w1 x)) * (w3 x)): the wave's ft 0-3 are w1 rows, ft 4-7 the same features of w3. Two values at a
    time; registers v[192:255]."""
    L = []
    n = 0
    for tt in range(nt):
        L += out_row(tt)
        for g in range(2):
            o = 192 + 4 * (n % 2)
            n += 1
            for p in range(4):                   # 2 values each
                ft, e = 2 * g + p // 2, (p % 2) * 2
                w = 208 + 16 * (p % 2)
                ga, gb, ua, ub, ta, tb, pk = w, w + 1, w + 2, w + 3, w + 4, w + 5, w + 6
                b1, b3 = (8 * ft + tt) * 4 + e, (8 * (ft + 4) + tt) * 4 + e
                L += [f"v_accvgpr_read_b32 v{ga}, a{b1}", f"v_accvgpr_read_b32 v{gb}, a{b1 + 1}",
                      f"v_accvgpr_read_b32 v{ua}, a{b3}", f"v_accvgpr_read_b32 v{ub}, a{b3 + 1}"]
                if w8:
                    L += [f"v_mul_f32 v{ga}, %[sc], v{ga}", f"v_mul_f32 v{gb}, %[sc], v{gb}",
                          f"v_mul_f32 v{ua}, %[su], v{ua}", f"v_mul_f32 v{ub}, %[su], v{ub}"]
                L += [f"v_cvt_pk_bf16_f32 v{ta}, v{ga}, v{gb}", f"v_cvt_pk_bf16_f32 v{tb}, v{ua}, v{ub}",
                      f"v_lshlrev_b32 v{ga}, 16, v{ta}", f"v_and_b32 v{gb}, 0xffff0000, v{ta}",
                      f"v_lshlrev_b32 v{ua}, 16, v{tb}", f"v_and_b32 v{ub}, 0xffff0000, v{tb}",
                      f"v_mul_f32 v{ta}, 0xbfb8aa3b, v{ga}", f"v_mul_f32 v{tb}, 0xbfb8aa3b, v{gb}",
                      f"v_exp_f32 v{ta}, v{ta}", f"v_exp_f32 v{tb}, v{tb}", "s_nop 0",
                      f"v_add_f32 v{ta}, 1.0, v{ta}", f"v_add_f32 v{tb}, 1.0, v{tb}",
                      f"v_rcp_f32 v{ta}, v{ta}", f"v_rcp_f32 v{tb}, v{tb}", "s_nop 0",
                      f"v_mul_f32 v{ta}, v{ga}, v{ta}", f"v_mul_f32 v{tb}, v{gb}, v{tb}",
                      f"v_cvt_pk_bf16_f32 v{pk}, v{ta}, v{tb}",
                      f"v_lshlrev_b32 v{ta}, 16, v{pk}", f"v_and_b32 v{tb}, 0xffff0000, v{pk}",
                      f"v_mul_f32 v{ta}, v{ta}, v{ua}", f"v_mul_f32 v{tb}, v{tb}, v{ub}",
                      f"v_cvt_pk_bf16_f32 v{o + p}, v{ta}, v{tb}"]
            L.append(f"buffer_store_dwordx4 {quad(o)}, v{ROW_VOFF}, %[ro], 0 offen offset:{64 * g}")
    return L


def partial_epilogue(nt=8):
    """The raw fp32 sums, straight from the accumulators: 16 bytes (4 features) per lane and store."""
    L = []
    for tt in range(nt):
        L += out_row(tt)
        for ft in range(8):
            b = (8 * ft + tt) * 4
            L.append(f"buffer_store_dwordx4 a[{b}:{b + 3}], v{ROW_VOFF}, %[ro], 0 offen offset:{(ft >> 1) * 128 + (ft & 1) * 16}")
    return L + ["s_nop 7"]


def part_epilogue():
    """The raw fp32 sums of a part of a tile, straight from the accumulators: 1 KiB per MFMA tile, 8 KiB per wave, token blocks
    outermost over all waves; token blocks without rows (%[part] - 1 of the wave's 8 have some) are left out."""
    L = [f"v_mov_b32 v{ROW_VOFF}, v{OUT_VOFF}"]
    for tt in range(8):
        L += [f"s_cmp_le_i32 %[part], {tt + 1}", "s_cbranch_scc1 31f"]
        for ft in range(8):
            b = (8 * ft + tt) * 4
            L.append(f"buffer_store_dwordx4 a[{b}:{b + 3}], v{ROW_VOFF}, %[ro], 0 offen offset:{1024 * (ft % 4)}")
            if ft % 4 == 3:
                L.append(f"v_add_u32 v{ROW_VOFF}, {0x1000 if ft == 3 else 0x7000:#x}, v{ROW_VOFF}")
    return L + ["31:", "s_nop 7"]


def gelu_drain(dt):
    """The pieces of the deferred tile with nothing to hide behind: token blocks 1 .. %[dnt] - 1, 4 pieces each, those of a block read
    back while the one before is worked on. v[192:255] free."""
    L = [f"v_mov_b32 v{ROW_VOFF}, v{DEF_ST}", f"v_mov_b32 v{DEF_LD}, v{SCR_VOFF}"]

    def back(tt):
        return [f"buffer_load_dwordx4 {quad(192 + 16 * (tt % 2) + 4 * g)}, v{DEF_LD}, %[scr], 0 offen offset:{1024 * g}" for g in range(4)]
    L += back(1)
    for tt in range(1, 8):
        if tt < 7:
            L += [f"s_cmp_le_i32 %[dnt], {tt + 1}", "s_cbranch_scc1 51f", f"v_add_u32 v{DEF_LD}, 0x1000, v{DEF_LD}"] + back(tt + 1)
            L += [f"s_waitcnt vmcnt({4 if tt == 1 else 8})", "s_branch 52f", "51:"]   # younger: the stores of the block before, these loads
        L += ["s_waitcnt vmcnt(0)", "52:", f"v_add_u32 v{ROW_VOFF}, {'%[dldo]' if tt > 1 else '%[dd]'}, v{ROW_VOFF}"]
        for g in range(4):
            L += [i for i, _ in gelu_words(dt, 192 + 16 * (tt % 2) + 4 * g, 224 + 4 * g, 4)]
            L.append(f"buffer_store_dwordx4 {quad(224 + 4 * g)}, v{ROW_VOFF}, %[dro], 0 offen offset:{64 * g}")
        if tt < 7:
            L += [f"s_cmp_le_i32 %[dnt], {tt + 1}", "s_cbranch_scc1 53f"]
    return L + ["53:", "s_nop 7"]


def tile(dt, w8, gelu, bias, epi, heights=HEIGHTS):
    """A tile of any height: the text of its number of token blocks, %[nt]. 16 bits: raw sums where it is a part of a tile, which has 8
    (%[part])."""
    texts = []
    for nt in heights:
        parts = nt == 8 and dt != "F8"
        L = [f"{100 + nt}:"] + k_loop(dt, w8, gelu, bias, nt)
        L += ["s_cmp_lg_u32 %[part], 0", "s_cbranch_scc1 41f"] if parts else []
        L += epi(nt)
        L += ["s_branch 199f", "41:"] + part_epilogue() if parts else []
        texts += L + ["s_branch 199f"]
    jumps = []
    for nt in heights[1:]:
        jumps += [f"s_cmp_eq_u32 %[nt], {nt}", f"s_cbranch_scc1 {100 + nt}f"]
    return jumps + texts[:-1] + ["199:"]


def check_trans(lines):
    """A transcendental result is read by another instruction at the earliest two instructions later."""
    import re
    for a, b in zip(lines, lines[1:]):
        mm = re.match(r"v_(exp|rcp)_f32 (v\d+),", a)
        if mm and re.search(rf"[ |\-]{mm.group(2)}\b", b.split(",", 1)[1] if "," in b else ""):
            raise AssertionError((a, b))


def generate():
    out = ["// Generated by gen_gemm4w.py; do not edit. See that script for the register map and the schedule.", ""]
    texts = []
    for dt, w8, gelu, bias in (("BF16", False, False, False), ("BF16", False, False, True), ("F16", False, False, True),
                               ("BF16", False, True, True), ("F16", False, True, True), ("BF16", True, False, False), ("BF16", True, False, True)):
        name = f"HDMOE_G4_TILE_{dt}{'_W8' if w8 else ''}{'_GELU' if gelu else '_BIAS' if bias else ''}"
        texts.append((name, tile(dt, w8, gelu, bias, lambda nt: epilogue(dt, w8, bias, gelu, nt))))
    for w8 in (False, True):
        texts.append((f"HDMOE_G4_TILE_BF16{'_W8' if w8 else ''}_SWIGLU", tile("BF16", w8, False, False, lambda nt: swiglu_epilogue(w8, nt))))
        texts.append((f"HDMOE_G4_TILE_BF16{'_W8' if w8 else ''}_PARTIAL", k_loop("BF16", w8, False, False) + partial_epilogue()))
    texts.append(("HDMOE_G4_FILL", reads(0, 0, False, 0)))
    texts.append(("HDMOE_G4_FILL_W8", reads(0, 0, True, 0) + ["s_waitcnt lgkmcnt(0)"] + [i for i, _ in conversions(0)]))
    for dt in ("BF16", "F16"):
        texts.append((f"HDMOE_G4_DRAIN_{dt}", DRAIN_WAIT + gelu_drain(dt)))
    for bias in (False, True):
        texts.append((f"HDMOE_G4_TILE_F8{'_BIAS' if bias else ''}", tile("F8", False, False, bias, lambda nt: epilogue("F8", False, bias, False, nt))))
    texts.append(("HDMOE_G4_TILE_F8_PARTIAL", tile("F8", False, False, False, partial_epilogue)))
    texts.append(("HDMOE_G4_FILL_F8", burst8(0)[0]))
    for name, lines in texts:
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

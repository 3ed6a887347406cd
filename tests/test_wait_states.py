"""Wait states that the hardware wants between two instructions and that hand-written statements have to keep themselves: the compiler
adds them between its own instructions, but neither inside a statement nor where one begins or ends. Every built kernel with such
statements is read back and each pair of instructions that can follow each other is looked at, over branches too."""
import os
import re
import subprocess

import pytest

from comfyui_amd import _lib
from tests.test_gemm4w_registers import OBJDUMP, code_objects

KERNELS = re.compile(r"(gemm4w_kernel|swiglu224_kernel|swiglu4w_kernel|grouped_gemm_kernel)")
TRANS = re.compile(r"v_(exp|log|rcp|rsq|sqrt|sin|cos)_")
REG = re.compile(r"\b([vas])(?:\[(\d+):(\d+)\]|(\d+)\b)|\b(vcc|m0|exec)\b")


def registers(text):
    out = set()
    for kind, lo, hi, one, named in REG.findall(text):
        if named:
            out.add(named)
        elif one:
            out.add(kind + one)
        else:
            out.update(f"{kind}{i}" for i in range(int(lo), int(hi) + 1))
    return out


class Instruction:
    __slots__ = ("op", "text", "operands", "target", "writes", "reads", "waits")

    def __init__(self, op, text, target):
        self.op, self.text, self.target = op, text, target
        self.operands = [o.strip() for o in re.split(r",(?![^\[]*\])", text)] if text else []
        self.waits = int(self.operands[0], 0) + 1 if op == "s_nop" else 1
        first = registers(self.operands[0]) if self.operands else set()
        rest = registers(" ".join(self.operands[1:]))
        store = op.startswith(("buffer_store", "global_store", "scratch_store", "ds_write", "s_cmp", "s_bitcmp", "s_waitcnt", "s_cbranch", "s_nop"))
        self.writes = set() if store else first
        self.reads = rest | (first if store else set())
        if op.endswith("_e32") and op.startswith(("v_cndmask", "v_addc", "v_subb")):
            self.reads.add("vcc")

    @property
    def valu(self):
        return self.op.startswith("v_") and not self.op.startswith("v_mfma")

    @property
    def vmem(self):
        return self.op.startswith(("buffer_", "global_", "scratch_"))

    @property
    def lane(self):
        return self.op.startswith(("v_readlane", "v_readfirstlane"))


def needed(a, b):
    """Wait states wanted between a and a later b."""
    n = 0
    if a.valu:
        scalars = {r for r in a.writes if r[0] == "s" or r == "vcc"}
        if b.lane and not a.lane and registers(b.operands[1]) & a.writes:
            n = max(n, 1)
        if scalars:
            if b.vmem and scalars & b.reads:
                n = max(n, 5)
            if b.valu and scalars & b.reads:
                n = max(n, 2)
            if b.op.startswith(("v_readlane", "v_writelane")) and registers(b.operands[2]) & scalars:
                n = max(n, 4)
        if TRANS.match(a.op) and b.valu and not TRANS.match(b.op) and a.writes & b.reads:
            n = max(n, 1)
        part = re.search(r"op_sel:\[[01],[01],1\]", a.text) or ("dst_sel" in a.text and "dst_sel:DWORD" not in a.text)
        if part and b.valu and a.writes & b.reads:
            n = max(n, 1)
    elif a.op.startswith("s_") and "m0" in a.writes:
        if b.vmem and b.text.endswith("lds"):
            n = max(n, 1)
    elif a.op.startswith("buffer_store_dwordx") and a.op[-1] in "34":
        offset = a.operands[3].split()[0]
        if not offset.startswith(("s", "m0")) and b.valu and registers(a.operands[0]) & b.writes:
            n = max(n, 1)
    return n


def interesting(a):
    if a.valu:
        return any(r[0] == "s" or r == "vcc" for r in a.writes) or any(r[0] == "v" for r in a.writes)
    return "m0" in a.writes or a.op.startswith("buffer_store_dwordx")


def kernels(text):
    name, body, at = None, [], {}
    for line in text.splitlines():
        head = re.match(r"[0-9a-f]+ <(\S+)>:", line)
        if head:
            if name:
                yield name, body, at
            name, body, at = (head.group(1) if KERNELS.search(head.group(1)) else None), [], {}
        elif name and "//" in line:
            code, _, note = line.partition("//")
            words = code.strip().split(None, 1)
            address = int(re.match(r"\s*([0-9A-F]+):", note).group(1), 16)
            target = re.search(r"<\S+?(?:\+0x([0-9a-f]+))?>$", note.strip()) if "branch" in words[0] else None
            if not body:
                start = address
            at[address - start] = len(body)
            body.append(Instruction(words[0], words[1] if len(words) > 1 else "", int(target.group(1) or "0", 16) if target else None))
    if name:
        yield name, body, at


def violations(body, at):
    found = []
    for i, a in enumerate(body):
        if not interesting(a):
            continue
        scalar = any(r[0] == "s" or r == "vcc" for r in a.writes)
        reach = 5 if a.valu and scalar else 1
        todo, seen = [(i + 1, 0)], set()
        while todo:
            j, states = todo.pop()
            if j >= len(body) or states >= reach or (j, states) in seen:
                continue
            seen.add((j, states))
            b = body[j]
            if needed(a, b) > states:
                found.append((a.op, a.text, b.op, b.text, states))
            if b.op in ("s_endpgm", "s_setpc_b64"):
                continue
            if b.target is not None:
                todo.append((at[b.target], states + 1))
            if b.op != "s_branch":
                todo.append((j + 1, states + b.waits))
    return found


@pytest.mark.skipif(not os.path.exists(OBJDUMP), reason="needs llvm-objdump")
def test_hand_written_statements_keep_the_wait_states(tmp_path):
    seen = set()
    for i, obj in enumerate(code_objects(_lib.LIB_PATH)):
        f = tmp_path / f"{i}.o"
        f.write_bytes(obj)
        text = subprocess.run([OBJDUMP, "-d", str(f)], capture_output=True, text=True, check=True).stdout
        for name, body, at in kernels(text):
            seen.add(KERNELS.search(name).group(1))
            assert not violations(body, at), (name, violations(body, at)[:5])
    assert len(seen) == 4


def test_the_rules_find_what_they_are_for():
    def pair(first, second, between=()):
        make = lambda line: Instruction(*(line.split(None, 1) + [""])[:2], None)
        body = [make(x) for x in (first, *between, second)]
        return violations(body, {})
    assert pair("v_mov_b32_e32 v0, v9", "v_readfirstlane_b32 s10, v0")              # the one that stored through a stale slot
    assert not pair("v_mov_b32_e32 v0, v9", "v_readfirstlane_b32 s10, v0", ["s_nop 0"])
    assert pair("v_readlane_b32 s4, v1, 3", "buffer_load_dwordx4 v[2:5], v6, s[4:7], 0 offen", ["s_nop 3"])
    assert not pair("v_readlane_b32 s4, v1, 3", "buffer_load_dwordx4 v[2:5], v6, s[4:7], 0 offen", ["s_nop 4"])
    assert pair("v_exp_f32_e32 v3, v4", "v_add_f32_e32 v5, 1.0, v3")
    assert not pair("v_exp_f32_e32 v3, v4", "v_add_f32_e32 v5, 1.0, v6")
    assert pair("s_add_u32 m0, s4, 0x1000", "buffer_load_dwordx4 v4, s[64:67], s5 offen lds")
    assert pair("buffer_store_dwordx4 v[34:37], v9, s[4:7], 0 offen", "v_mov_b32_e32 v35, 0")
    assert not pair("buffer_store_dwordx4 v[34:37], v9, s[4:7], s8 offen", "v_mov_b32_e32 v35, 0")

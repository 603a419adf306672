"""Registers that an inline-assembly statement of the device code writes or reads closer to the instruction that reads or
wrote them than the hardware allows, looked for in the assembly of the library's own kernels, built as the library is.

The compiler fills these distances with s_nop between its own instructions.  It takes an inline-assembly statement for no
vector instruction, so that before, after and inside of one the source has to keep them.  In instructions that lie
between the two (s_nop counts as its operand + 1):
  2  a vector instruction writes a scalar register, vcc among them; a vector instruction reads it
  4  the same; a lane move takes it as its lane
  5  the same; a memory access takes it as its base
  1  a vector instruction writes a vector register; v_readlane, v_readfirstlane read it
  2  the same; a DPP operand reads it
  1  a transcendental function's result is read by another vector instruction
  1  a vector instruction writes the registers that a store of more than 64 bits stores
"""
import os
import re
import shutil
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "bps_nav_amd", "csrc")

REG = re.compile(r"^(-|\|)*([vs])(?:(\d+)|\[(\d+):(\d+)\])(\|)?$")
TRANS = re.compile(r"v_(rcp|rsq|sqrt|exp|log|sin|cos)_")
REACH = 5


class Ins:
    def __init__(self, text, asm, at):
        self.text, self.asm, self.at = text, asm, at
        self.op, _, rest = text.partition(" ")
        # modifiers follow the last operand without a comma
        self.args = [a.strip().split(" ")[0] for a in rest.split(",")] if rest else []
        self.dpp = "_dpp" in self.op or " quad_perm:" in rest or " row_" in rest or " wave_" in rest
        sets = [registers(a) for a in self.args]
        n = 0
        if self.vector():
            n = 2 if "_co_" in self.op or "div_scale" in self.op else 1
        self.writes = set().union(*sets[:n]) if n else set()
        self.reads = set().union(*sets[n:]) if sets[n:] else set()
        if self.op.startswith(("v_writelane", "v_fmac", "v_mac")):
            self.reads |= self.writes

    def vector(self):
        return self.op.startswith("v_")

    def memory(self):
        return self.op.startswith(("global_", "flat_", "buffer_", "scratch_"))

    def waits(self):
        return int(self.args[0], 0) + 1 if self.op == "s_nop" else 1


def registers(arg):
    if arg in ("vcc", "exec"):
        return {arg + "_lo", arg + "_hi"}
    if arg in ("vcc_lo", "vcc_hi", "exec_lo", "exec_hi", "m0"):
        return {arg}
    m = REG.match(arg)
    if not m:
        return set()
    lo = int(m.group(3) or m.group(4))
    return {m.group(2) + str(i) for i in range(lo, int(m.group(5) or lo) + 1)}


def scalars(regs):
    return {r for r in regs if r[0] == "s" or r.startswith("vcc")}


def vectors(regs):
    return {r for r in regs if r[0] == "v" and not r.startswith("vcc")}


def needed(a, b):
    """(distance, registers) that `b` has to keep from `a`, for every rule that joins the two."""
    if a.vector():
        s, v = scalars(a.writes), vectors(a.writes)
        if b.vector():
            lane = registers(b.args[2]) if b.op.startswith(("v_readlane", "v_writelane")) else set()
            yield 4, s & lane
            yield 2, s & (b.reads - lane)
            if b.op.startswith(("v_readlane", "v_readfirstlane")):
                yield 1, v & registers(b.args[1])
            if b.dpp:
                yield 2, v & registers(b.args[1])
            if TRANS.match(a.op) and not TRANS.match(b.op):
                yield 1, v & b.reads
        if b.memory():
            yield 5, s & b.reads
    elif a.memory() and "store" in a.op and b.vector():
        for arg in a.args:
            stored = vectors(registers(arg))
            if len(stored) > 2:
                yield 1, stored & b.writes


def functions(lines):
    """[(name, [Ins], {label: index})]"""
    out, asm, name, body, labels = [], False, None, [], {}
    for at, line in enumerate(lines, 1):
        if "ASMSTART" in line:
            asm = True
            continue
        if "ASMEND" in line:
            asm = False
            continue
        line = line.split(";")[0].strip()
        if not line:
            continue
        if line.endswith(":"):
            if not line.startswith(".L") and not line[0].isdigit():
                if name and body:
                    out.append((name, body, labels))
                name, body, labels = line[:-1], [], {}
            elif line[0].isdigit():   # a label of an inline statement: its branches name it by 1b or 2f
                labels.setdefault(line[:-1], []).append(len(body))
            else:
                labels[line[:-1]] = len(body)
            continue
        if line.startswith(".") or not name:
            continue
        body.append(Ins(re.sub(r"\s+", " ", line), asm, at))
    if name and body:
        out.append((name, body, labels))
    return out


def too_close(text):
    """[(function, line, instruction, line, instruction, distance, wanted)], both ends' lines in the text"""
    found = []
    for name, body, labels in functions(text.splitlines()):
        came = {}   # index -> branches that lead there
        for i, ins in enumerate(body):
            if not ins.op.startswith(("s_branch", "s_cbranch")) or not ins.args:
                continue
            t = ins.args[0]
            if re.fullmatch(r"\d+[bf]", t):
                places = labels.get(t[:-1], [])
                to = [p for p in places if p <= i][-1:] if t[-1] == "b" else [p for p in places if p > i][:1]
            else:
                to = [labels[t]] if t in labels else []
            for p in to:
                came.setdefault(p, []).append(i)

        def back(i, dist, end, seen):
            """instructions before i, `dist` of distance between them and `end`"""
            before = list(came.get(i, ()))
            if i > 0 and not body[i - 1].op.startswith(("s_branch", "s_endpgm", "s_setpc")):
                before.append(i - 1)
            for j in before:
                if (j, dist) in seen:
                    continue
                seen.add((j, dist))
                a = body[j]
                if a.asm or end.asm:
                    for want, regs in needed(a, end):
                        if regs and dist < want:
                            found.append((name, a.at, a.text, end.at, end.text, dist, want))
                d = dist + a.waits()
                if d < REACH:
                    back(j, d, end, seen)

        for i, ins in enumerate(body):
            if ins.vector() or ins.memory():
                back(i, 0, ins, set())
    return found


ASM = "\t;;#ASMSTART\n\t%s\n\t;;#ASMEND\n"


# (instructions, s_nop count between them that is enough).  The first or the second is the inline statement.
@pytest.mark.parametrize("first, second, enough", [
    ("v_cmp_ne_u32_e64 s[14:15], s7, v57", "v_cndmask_b32_e64 v2, v3, v2, s[14:15]", 2),
    ("v_cmp_ne_u32_e32 vcc, 0, v57", "v_cndmask_b32_e32 v2, v3, v2, vcc", 2),
    ("v_readfirstlane_b32 s4, v1", "v_add_u32_e32 v2, s4, v2", 2),
    ("v_readfirstlane_b32 s4, v1", "v_readlane_b32 s6, v2, s4", 4),
    ("v_readfirstlane_b32 s5, v1", "global_store_dword v2, v3, s[4:5]", 5),
    ("v_mul_u32_u24_e32 v1, s2, v1", "v_readlane_b32 s6, v1, 3", 1),
    ("v_mul_u32_u24_e32 v1, s2, v1", "v_mov_b32_dpp v2, v1 quad_perm:[1,0,3,2] row_mask:0xf bank_mask:0xf", 2),
    ("v_rsq_f32_e32 v1, v2", "v_mul_f32_e32 v3, v1, v2", 1),
    ("global_store_dwordx4 v1, v[4:7], s[2:3]", "v_mov_b32_e32 v6, 0", 1),
])
def test_the_reader_sees_every_rule(first, second, enough):
    for inline in (0, 1):
        for nop in range(enough + 1):
            a, b = (ASM % x if inline == k else f"\t{x}\n" for k, x in enumerate((first, second)))
            between = f"\ts_nop {nop - 1}\n" if nop else ""
            assert bool(too_close(f"f:\n{a}{between}{b}\ts_endpgm\n")) == (nop < enough), (first, second, nop)
    # the compiler's own pair is its own business; a way there through a branch counts
    assert not too_close(f"f:\n\t{first}\n\t{second}\n\ts_endpgm\n")
    if enough >= 2:
        assert too_close(f"f:\n\t{first}\n\ts_cbranch_scc1 .L1\n\ts_nop 7\n.L1:\n{ASM % second}\ts_endpgm\n")


@pytest.mark.skipif(shutil.which("hipcc") is None and not os.path.exists("/opt/rocm/bin/hipcc"), reason="needs the compiler")
def test_the_kernels_keep_the_distances(tmp_path):
    out = str(tmp_path / "kernels.s")
    line = subprocess.run(["make", "-C", CSRC, "-n", "-B", "kernels.o"], check=True, capture_output=True, text=True).stdout
    cmd = [c for c in line.splitlines() if "hipcc" in c and "kernels.hip" in c][0].split()
    cmd = cmd[:cmd.index("-c")] + ["--cuda-device-only", "-S", "kernels.hip", "-o", out]
    subprocess.run(cmd, check=True, cwd=CSRC, stderr=subprocess.DEVNULL)
    with open(out) as f:
        text = f.read()
    assert text.count("ASMSTART") > 1000 and len(functions(text.splitlines())) > 10
    found = too_close(text)
    assert not found, "\n".join(f"{n[:60]}: '{a}' (line {i}), {d} of {w} before '{b}' (line {j})" for n, i, a, j, b, d, w in found)

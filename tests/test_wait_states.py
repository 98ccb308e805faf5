"""Wait states of the BM kernels' compiled gfx950 assembly.

The hardware does not interlock some pairs of vector instructions; the compiler
puts other instructions or s_nop between them, but it does not look inside inline
assembly.  Here every kernel that uses the assembly blocks of bm_device.h is
compiled and each pair is checked, wherever its two halves come from:

* a VGPR that a vector instruction wrote, read by v_readlane or v_readfirstlane:
  one wait state between;
* the same, read through DPP: two;
* an SGPR (or VCC) that a vector instruction wrote, read by a vector
  instruction: two; as the lane of v_readlane or v_writelane: four; by a memory
  instruction: five;
* the result of a transcendental instruction, read by another kind of vector
  instruction: one.

A reduction's assembly block must leave nothing that depends on what the
compiler places next: readers of its results are also put right behind it.

Instructions are followed in the order of the listing, so a pair across the
back edge of a loop is not seen; the blocks' loops begin and end such that their
own back edges hold no pair (an s_nop or three scalar instructions).  A wrong
value here would change step control, and with it the number of barriers that
the waves of a block meet."""
import os
import re
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "cochlearmodel_amd", "csrc")
TRANS = re.compile(r"v_(rcp|rsq|sqrt|log|exp|sin|cos)_")


def _assembly(src, out):
    hipcc = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
    if not os.path.exists(hipcc):
        pytest.skip("hipcc not available")
    cmd = [hipcc, "--offload-arch=gfx950", "-O3", "-std=c++17", "-ffp-contract=off", "-Xclang", "-target-feature",
           "-Xclang", "-packed-fp32-ops", "-I", CSRC, "-I", os.path.join(ROOT, "include"), "--cuda-device-only", "-S",
           os.path.join(CSRC, src), "-o", str(out)]
    r = subprocess.run(cmd, capture_output=True, text=True)
    assert r.returncode == 0, r.stderr[-2000:]
    return out.read_text()


def _regs(operand):
    """Registers of an operand: {("v", 3), ("v", 4)} of v[3:4]."""
    operand = operand.strip().strip("-|")
    if operand == "vcc":
        return {("s", "vcc")}
    m = re.match(r"([vsa])\[(\d+):(\d+)\]$", operand)
    if m:
        return {(m.group(1), k) for k in range(int(m.group(2)), int(m.group(3)) + 1)}
    m = re.match(r"([vsa])(\d+)(?!\w)", operand)
    return {(m.group(1), int(m.group(2)))} if m else set()


def _parse(line):
    """(mnemonic, written registers, operand strings read) of a vector or memory instruction."""
    mn, _, rest = line.partition(" ")
    ops = [o.strip() for o in re.split(r",\s*", rest.strip())] if rest else []
    n_dst = 1
    if re.match(r"v_(add_co|sub_co|subrev_co|addc_co|subb_co|div_scale|mad_u64_u32|mad_i64_i32)", mn):
        n_dst = 2
    dst, src = ops[:n_dst], ops[n_dst:]
    if mn.startswith("v_cmpx") or mn.startswith("v_nop"):
        dst, src = [], ops
    written = set().union(*(_regs(o) for o in dst)) if dst else set()
    if re.match(r"v_(fmac|fma_mix|mac|pk_fmac|dot2c|swap)", mn) or mn.startswith("v_mov_b32_dpp"):
        src = src + dst[:1]
    return mn, written, src


def _violations(lines):
    """Pairs too close together in a straight listing of instructions."""
    found = []
    recent = []   # (age, mnemonic, written) of the last vector instructions, age in wait states
    for k, line in enumerate(lines):
        mn = line.split(" ")[0]
        if mn == "s_nop":
            wait = int(line.split()[1], 0) + 1
            recent = [(a + wait, m, w) for a, m, w in recent if a + wait < 6]
            continue
        vector = mn.startswith("v_")
        memory = mn.startswith(("global_", "buffer_", "flat_", "scratch_"))
        written = set()
        if vector or memory:
            if vector:
                _, written, src = _parse(line)
            else:
                src = [o.strip() for o in re.split(r",\s*", line.partition(" ")[2])]
            dpp = "_dpp" in mn
            read = set().union(*(_regs(o.split(" ")[0]) for o in src)) if src else set()
            src0 = _regs(src[0].split(" ")[0]) if src else set()
            if dpp and mn.startswith("v_fmac"):
                through = _regs(src[0].split(" ")[0])
            else:
                through = src0 if dpp else set()
            lane = mn.startswith(("v_readlane", "v_readfirstlane"))
            for age, m, w in recent:
                v = {r for r in w if r[0] == "v"}
                s = {r for r in w if r[0] == "s"}
                if lane and age < 1 and v & src0:
                    found.append(("readlane of a fresh VGPR", k, m, line))
                if age < 2 and v & through:
                    found.append(("DPP read of a fresh VGPR", k, m, line))
                if vector and age < 2 and s & read:
                    found.append(("vector read of a fresh SGPR", k, m, line))
                if mn.startswith(("v_readlane", "v_writelane")) and age < 4 and s & _regs(src[-1].split(" ")[0]):
                    found.append(("lane select of a fresh SGPR", k, m, line))
                if memory and age < 5 and s & read:
                    found.append(("memory read of a fresh SGPR", k, m, line))
                if vector and age < 1 and TRANS.match(m) and not TRANS.match(mn) and v & read:
                    found.append(("fresh transcendental result", k, m, line))
        recent = [(a + 1, m, w) for a, m, w in recent if a + 1 < 6]
        if vector:
            recent.append((0, mn, written))
    return found


def _instructions(text):
    lines = [l.split(";")[0].strip().replace("\t", " ") for l in text.split("\n")]
    return [l for l in lines if l and not l.startswith((".", "/")) and not l.endswith(":")]


def _functions(asm):
    for m in re.finditer(r"\n(_ZN?\w+):", asm):
        text = asm[m.end():asm.find(".Lfunc_end", m.end())]
        blocks = re.findall(r";;#ASMSTART(.*?);;#ASMEND", text, re.S)
        yield m.group(1), _instructions(text), [_instructions(b) for b in blocks if "row_half_mirror" in b]


def _readers(block):
    """An instruction that reads each register the block wrote."""
    out = []
    for kind, num in sorted(set().union(*(_parse(l)[1] for l in block if l.startswith("v_")))):
        out.append(f"v_readlane_b32 s200, v{num}, 0" if kind == "v" else f"v_mov_b32_e32 v255, s{num}")
    return out


def test_the_check_sees_each_kind_of_pair():
    assert _violations(["v_add_f32_dpp v1, v1, v1 row_mirror", "s_cmp_gt_i32 s1, 0", "v_readlane_b32 s0, v1, 0"]) == []
    bad = [["v_add_f32_dpp v1, v2, v2 row_mirror", "v_readlane_b32 s0, v1, 0"],
           ["v_mul_f32_e32 v1, v2, v3", "s_nop 0", "v_add_f32_dpp v4, v1, v5 row_mirror"],
           ["v_readlane_b32 s0, v1, 63", "s_nop 0", "v_mul_f32_e32 v2, s0, v3"],
           ["v_cmp_gt_f32_e32 vcc, v1, v2", "v_cndmask_b32_e32 v1, v2, v3, vcc"],
           ["v_readfirstlane_b32 s4, v1", "s_nop 2", "global_load_dword v1, v2, s[4:5]"],
           ["v_rcp_f32_e32 v1, v2", "v_mul_f32_e32 v3, v1, v1"]]
    for lines in bad:
        assert len(_violations(lines)) == 1, lines
        assert _violations([lines[0], "s_nop 7", lines[-1]]) == []


@pytest.mark.parametrize("src", ["bm_split_kernel.hip", "bm_kernel.hip"])
def test_wait_states(src, tmp_path):
    asm = _assembly(src, tmp_path / "k.s")
    n = lanes = trees = 0
    for name, lines, blocks in _functions(asm):
        n += len(lines)
        trees += len(blocks)
        lanes += sum(l.startswith("v_readlane") for l in lines)
        bad = _violations(lines)
        assert not bad, (name, len(bad), bad[:5])
        for block in blocks:
            for reader in _readers(block):
                assert not _violations(block + [reader]), (name, block, reader)
    assert n > 10000 and lanes > 50 and trees > 20

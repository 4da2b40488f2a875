"""Wait states in the built kernels.  The compiler keeps them between instructions of its
own but not for inline assembly: a statement that reads what a lane read or a vector
instruction has just written has to keep them itself.  Checked in the disassembly: between
the vector instruction that writes a register and the one that reads it lie 2 wait states
for an SGPR, 2 for a VGPR read by DPP or permlane, 1 for a VGPR read by readlane."""
import os
import re
import shutil
import subprocess

import pytest

import blockstructuredsolvers_amd as bss

LIB = os.path.join(os.path.dirname(bss.__file__), "libbss.so")
OBJDUMP = "/opt/rocm/lib/llvm/bin/llvm-objdump"
REG = re.compile(r"\b([vs])(?:(\d+)|\[(\d+):(\d+)\])")


def regs(text):
    out = set()
    for k, one, lo, hi in REG.findall(text):
        out.update((k, r) for r in (range(int(lo), int(hi) + 1) if lo else [int(one)]))
    return out


def hazards(lines):
    """(instruction, the ones before it) of every pair that is too close, in straight-line
    order"""
    found, past = [], []  # past: (wait states, registers written, text), newest last
    for line in lines:
        text = line.split("//")[0].strip()
        op, _, rest = text.partition(" ")
        if not text or text.endswith(":"):
            past = []
            continue
        if op == "s_nop":
            past = past[-3:] + [(int(rest, 0) + 1, set(), text)]
            continue
        if not op.startswith("v_"):
            past = past[-3:] + [(1, set(), text)]
            continue
        dst, _, src = rest.partition(",")
        writes, reads = regs(dst), regs(src)
        need_v = 0
        if op.startswith(("v_readlane", "v_readfirstlane")):
            need_v = 1
        elif op.startswith("v_permlane"):
            need_v = 2
            if "swap" in op:  # both operands are read and written
                writes = reads = regs(rest)
        elif "row_" in rest or "quad_perm" in rest:  # DPP: the first source
            need_v = 2
            reads = regs(src.split(",")[0]) | {r for r in reads if r[0] == "s"}
        elif op.startswith("v_mfma"):  # their results have longer waits of their own
            writes = set()
        for need, kind in ((2, "s"), (need_v, "v")):
            want = {r for r in reads if r[0] == kind}
            if any(w & want for w in recent(past, need)):
                found.append((text, [p[2] for p in past]))
        past = past[-3:] + [(1, writes, text)]
    return found


def recent(past, need):
    """what the instructions within `need` wait states before this one write"""
    for states, writes, _ in reversed(past):
        if need <= 0:
            return
        yield writes
        need -= states


def test_check_finds_a_close_pair():
    ok = ["v_readlane_b32 s3, v1, 5", "s_nop 1", "v_writelane_b32 v2, s3, 15"]
    assert not hazards(ok)
    for gap in ([], ["s_nop 0"], ["v_mov_b32 v7, v8"]):
        assert hazards([ok[0]] + gap + [ok[2]])
    assert hazards(["v_mul_f64 v[4:5], v[0:1], v[2:3]", "v_readlane_b32 s0, v5, 14"])
    dpp = "v_fmac_f64_dpp v[8:9], v[4:5], v[6:7] row_newbcast:3 row_mask:0xf bank_mask:0xf"
    assert hazards(["v_mul_f64 v[4:5], v[0:1], v[2:3]", "s_nop 0", dpp])
    assert not hazards(["v_mul_f64 v[6:7], v[0:1], v[2:3]", dpp])


def test_kernels_keep_wait_states(tmp_path):
    if not (os.path.exists(OBJDUMP) and os.path.exists(LIB)):
        pytest.skip("needs the built library and llvm-objdump")
    shutil.copy(LIB, tmp_path / "libbss.so")
    subprocess.run([OBJDUMP, "--offloading", "libbss.so"], cwd=tmp_path, check=True,
                   stdout=subprocess.DEVNULL)
    objects = sorted(p for p in tmp_path.iterdir() if "gfx950" in p.name)
    assert objects
    seen = 0
    for p in objects:
        out = subprocess.run([OBJDUMP, "-d", "--no-show-raw-insn", "--no-leading-addr", str(p)],
                             check=True, capture_output=True, text=True).stdout
        lines = out.splitlines()
        seen += len(lines)
        bad = hazards(lines)
        assert not bad, (p.name, len(bad), bad[:3])
    assert seen > 100000

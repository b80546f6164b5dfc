"""The built gfx950 code keeps the wait states that the hardware leaves to software around loads into LDS (CPU: the
library's own kernels, disassembled). The compiler inserts them for the instructions it selects, but not inside inline
assembly or between inline assembly and its neighbours:
  * a load into LDS reads M0 at least 1 wait state after a scalar write of M0;
  * a vector memory instruction reads an SGPR at least 5 wait states after a VALU instruction wrote it.
"""
import os
import re
import shutil
import subprocess

import pytest

from rustingstrata_amd import build

OBJDUMP = "/opt/rocm/llvm/bin/llvm-objdump"


def sgprs(text):
    out = set()
    for a, b, c in re.findall(r"\bs\[(\d+):(\d+)\]|\bs(\d+)\b", text):
        out.update(range(int(a), int(b) + 1) if a else [int(c)])
    return out


def short_waits(lines):
    """[(kernel, instruction, what, wait states)] of the places that wait too little, in program order."""
    bad, kernel, at, m0, valu, n_lds = [], "", 0, -10, {}, 0
    for line in lines:
        head = re.match(r"^[0-9a-f]+ <(.*)>:", line)
        if head:
            kernel, m0, valu = head.group(1), at - 10, {}
            continue
        line = line.split("//")[0].strip()
        if not re.match(r"^[a-z]+_", line):
            continue
        op, _, args = line.partition(" ")
        dst, _, src = args.partition(",")
        if op == "s_nop":
            at += int(args, 0) + 1
            continue
        if op.startswith(("global_", "buffer_", "scratch_", "flat_")):
            for r in sgprs(args):
                if at - valu.get(r, at - 10) - 1 < 5:
                    bad.append((kernel, line, f"s{r} written by a VALU instruction", at - valu[r] - 1))
            if "lds" in line:
                n_lds += 1
                if at - m0 - 1 < 1:
                    bad.append((kernel, line, "M0", at - m0 - 1))
        elif op.startswith("s_") and re.match(r"m0\b", dst):
            m0 = at
        elif op.startswith("s_"):
            for r in sgprs(dst):
                valu.pop(r, None)
        elif op.startswith("v_"):
            for r in sgprs(dst) | (sgprs(src.partition(",")[0]) if "_co_" in op or "div_scale" in op else set()):
                valu[r] = at
        at += 1
    return bad, n_lds


def test_the_scan_sees_short_waits():
    code = ["0000 <k>:", "s_mov_b32 m0, s4", "global_load_lds_dwordx4 v0, s[6:7]", "v_readfirstlane_b32 s7, v1",
            "s_mov_b32 m0, s4", "s_nop 0", "global_load_lds_dwordx4 v0, s[6:7]", "v_readfirstlane_b32 s8, v1",
            "s_mov_b64 s[6:7], s[8:9]", "global_load_dword v0, v1, s[6:7]"]
    bad, n = short_waits(code)
    assert n == 2 and [(b[2], b[3]) for b in bad] == [("M0", 0), ("s7 written by a VALU instruction", 2)]


@pytest.mark.skipif(not os.path.exists(OBJDUMP), reason="no llvm-objdump")
def test_loads_into_lds_keep_their_wait_states(tmp_path):
    if not os.path.exists(build.OUT):
        build.build()
    lib = shutil.copy(build.OUT, tmp_path)  # (the code objects are extracted beside the file)
    subprocess.run([OBJDUMP, "--offloading", lib], check=True, capture_output=True)
    objs = sorted(f for f in os.listdir(tmp_path) if f.endswith("gfx950"))
    assert objs
    total = 0
    for f in objs:
        text = subprocess.run([OBJDUMP, "-d", "--no-show-raw-insn", os.path.join(tmp_path, f)], check=True, capture_output=True,
                              text=True).stdout
        bad, n = short_waits(text.splitlines())
        total += n
        assert not bad, (f, len(bad), bad[:4])
    assert total > 0


def test_inline_assembly_computes_nothing():
    """Arithmetic stays in forms that the compiler selects instructions for: it knows the wait states between a
    transcendental result, a VALU write and an MFMA that reads it, but none of them for inline assembly."""
    for f in sorted(os.listdir(build.CSRC)):
        src = re.sub(r"//[^\n]*", "", open(os.path.join(build.CSRC, f)).read())
        for body in re.findall(r"\basm\s*(?:volatile\s*)?\(\s*((?:\"[^\"]*\"\s*)+)", src):
            assert not re.search(r"\bv_\w+", body), (f, body)

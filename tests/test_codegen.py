"""The gfx950 code of the built library: the waits that the hardware does not
make by itself and that the compiler does not add around inline assembly (its
hazard pass takes an asm block as one instruction), and no register spilled to
memory.  CPU only: ROCm's binary tools over the library built here from source."""
from __future__ import annotations

import glob
import os
import re
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
LIB = os.path.join(ROOT, "tailorquantkernel_amd", "libtqhip.so")
OBJDUMP = "/opt/rocm/llvm/bin/llvm-objdump"
READELF = "/opt/rocm/llvm/bin/llvm-readelf"
needs_tools = pytest.mark.skipif(not (os.path.exists(OBJDUMP) and os.path.exists(READELF)),
                                 reason="needs ROCm's llvm-objdump and llvm-readelf")


def scalar_regs(text: str) -> set[str]:
    """SGPR names (and m0, vcc) an operand text covers."""
    regs = {f"s{i}" for a, b in re.findall(r"\bs\[(\d+):(\d+)\]", text) for i in range(int(a), int(b) + 1)}
    return regs | set(re.findall(r"\b(?:s\d+|m0|vcc)\b", text))


def hazards(lines: list[str]) -> tuple[int, list[str]]:
    """(copies into LDS, those issued too early).  A scalar write of M0 has to
    be at least one wait state before a copy into LDS, which takes its address
    from M0; a vector write of an SGPR five before a memory instruction with
    that SGPR as its base."""
    copies, bad = 0, []
    code = [s for s in (line.split("//")[0].strip() for line in lines) if s and not s.endswith(":")]
    for i, ins in enumerate(code):
        if "_load_lds_" not in ins and not (ins.startswith("buffer_load") and ins.endswith(" lds")):
            continue
        copies += 1
        base = scalar_regs(ins.split(None, 1)[1])
        states = 0
        for prev in reversed(code[max(0, i - 5):i]):
            ops = prev.split(None, 1)
            if states >= 5:
                break
            if len(ops) == 2:
                dst = scalar_regs(ops[1].split(",")[0])
                if "_co_" in ops[0]:
                    dst |= scalar_regs(ops[1].split(",")[1])
                if (states < 1 and "m0" in dst) or (ops[0].startswith("v_") and dst & base):
                    bad.append(f"{prev} | {ins}")
                    break
            states += int(ops[1]) + 1 if ops[0] == "s_nop" else 1
    return copies, bad


def test_hazard_scan():
    load = "global_load_lds_dwordx4 v2, s[4:5]"
    assert hazards(["s_add_u32 m0, s1, 0x400", load]) == (1, [f"s_add_u32 m0, s1, 0x400 | {load}"])
    assert hazards(["s_mov_b32 m0, s1", "s_nop 0", load]) == (1, [])
    assert hazards(["v_readfirstlane_b32 s5, v9", "s_mov_b32 m0, s1", "s_nop 2", load])[1]
    assert hazards(["v_readfirstlane_b32 s5, v9", "s_mov_b32 m0, s1", "s_nop 3", load]) == (1, [])
    assert hazards(["v_readfirstlane_b32 s6, v9", "s_mov_b32 m0, s6", "s_nop 0", load]) == (1, [])


@pytest.fixture(scope="module")
def objects(tmp_path_factory):
    """The library's gfx950 code objects, one per source file."""
    tmp = tmp_path_factory.mktemp("codegen")
    shutil.copy(LIB, tmp / "lib.so")
    subprocess.run([OBJDUMP, "--offloading", "lib.so"], cwd=tmp, check=True, stdout=subprocess.DEVNULL)
    return sorted(glob.glob(str(tmp / "*gfx950")))


@needs_tools
def test_copies_into_lds_wait_for_their_operands(objects):
    copies, bad = 0, []
    for obj in objects:
        asm = subprocess.run([OBJDUMP, "-d", "--no-show-raw-insn", "--no-leading-addr", obj],
                             check=True, capture_output=True, text=True).stdout
        n, b = hazards(asm.splitlines())
        copies += n
        bad += b
    assert copies > 0, "no copy into LDS found: the scan no longer reads the code"
    assert not bad, f"{len(bad)} of {copies} copies, first: {bad[0]}"


@needs_tools
def test_no_kernel_spills(objects):
    kernels, spilled = 0, []
    for obj in objects:
        notes = subprocess.run([READELF, "--notes", obj], check=True, capture_output=True, text=True).stdout
        for name, n in re.findall(r"\.symbol: +(\S+?)\.kd.*?\.vgpr_spill_count: +(\d+)", notes, re.S):
            kernels += 1
            if int(n):
                spilled.append((name, int(n)))
    assert kernels > 100, "the kernels' notes are not read"
    assert not spilled, spilled

"""The direct L2 -> LDS loads of the built kernels, read back from the library's gfx950 code.

Such a load takes its LDS base from M0, and the instruction set asks for one wait state
between a scalar write of M0 and the load.  The compiler keeps that distance for its own
instructions but inserts nothing inside inline asm, where the library issues all of its
loads; too early a load may use the M0 before, and put its data at another LDS address
without any error.  Likewise a scalar base address written by the vector unit
(v_readfirstlane, v_readlane) needs five wait states before a vector memory instruction
reads it.
"""
from __future__ import annotations

import re
import shutil
import subprocess
from pathlib import Path

import pytest

LIB = Path(__file__).resolve().parents[1] / "mini-qwen-llm_amd" / "mqk" / "libmqk.so"
OBJDUMP = Path("/opt/rocm/llvm/bin/llvm-objdump")


def hazards(lines):
    """(number of LDS loads, the offending (instruction before, load) pairs) of an assembly listing."""
    loads, bad, before = 0, [], []
    for line in lines:
        if line.rstrip().endswith(">:"):  # the next function
            before = []
            continue
        if not line.startswith(("\t", " ")):
            continue
        ins = line.split("//")[0].strip()
        if not ins:
            continue
        if "lds_dword" in ins:
            loads += 1
            base = re.search(r"s\[(\d+):(\d+)\]", ins)
            distance = 0
            for prev in reversed(before[-6:]):
                if distance < 1 and re.match(r"s_\w+ m0,", prev):
                    bad.append((prev, ins))
                vector = re.match(r"v_read(?:firstlane|lane)_b32 s(\d+)", prev)
                if base and vector and distance < 5 and int(base[1]) <= int(vector[1]) <= int(base[2]):
                    bad.append((prev, ins))
                nop = re.match(r"s_nop (\w+)", prev)
                distance += int(nop[1], 0) + 1 if nop else 1
        before = (before + [ins])[-6:]
    return loads, bad


def test_the_scan_finds_a_missing_wait_state():
    early = ["\ts_mov_b32 m0, s4\n", "\tglobal_load_lds_dwordx4 v[2:3], off\n"]
    assert hazards(early) == (1, [("s_mov_b32 m0, s4", "global_load_lds_dwordx4 v[2:3], off")])
    assert hazards([early[0], "\ts_nop 0\n", early[1]]) == (1, [])
    base = ["\tv_readfirstlane_b32 s7, v1\n", "\ts_nop 3\n", "\tglobal_load_lds_dwordx4 v2, s[6:7]\n"]
    assert len(hazards(base)[1]) == 1
    assert hazards([base[0], "\ts_nop 4\n", base[2]]) == (1, [])


@pytest.mark.skipif(not LIB.exists() or not OBJDUMP.exists(), reason="needs the built library and llvm-objdump")
def test_loads_keep_their_wait_states(tmp_path):
    lib = tmp_path / LIB.name
    shutil.copy(LIB, lib)  # (the code objects are written beside it)
    subprocess.run([OBJDUMP, "--offloading", lib], check=True, capture_output=True)
    loads = 0
    for obj in sorted(tmp_path.glob("*gfx950")):
        text = subprocess.run([OBJDUMP, "-d", "--no-show-raw-insn", obj], check=True, capture_output=True, text=True).stdout
        n, bad = hazards(text.splitlines(keepends=True))
        loads += n
        assert not bad, f"{obj.name}: {len(bad)} loads, first {bad[0]}"
    assert loads > 0

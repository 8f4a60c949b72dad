"""The wait states the inline-asm copies of the GEMM kernels rely on (csrc/gemm_common.h, buf2lds_inner): no VALU
instruction may write an SGPR operand of a `buffer_load ... lds` in the five wait states before it, and a write of M0
must be one wait state ahead.  The compiler does not track either for inline asm, so the built library is checked, in
program order."""
import os
import re
import shutil
import subprocess

import pytest

from trenowanie_generatora_obrazkow_amd import _lib

OBJDUMP = "/opt/rocm/llvm/bin/llvm-objdump"


def _sgprs(operand):
    m = re.match(r"s\[(\d+):(\d+)\]$", operand)
    if m:
        return set(range(int(m[1]), int(m[2]) + 1))
    m = re.match(r"s(\d+)$", operand)
    return {int(m[1])} if m else set()


def hazards(lines):
    """(copies seen, [(line number, text)] of the copies that break a rule)."""
    since = {}  # SGPR -> wait states since a VALU instruction wrote it
    m0, copies, bad = 99, 0, []
    for i, line in enumerate(lines):
        text = line.split("//")[0].strip()
        if not re.match(r"(s|v|ds|buffer|global|flat|scratch)_\w+", text):
            continue
        op, _, rest = text.partition(" ")
        ops = [o.strip() for o in rest.split(",")]
        if op.startswith("buffer_load") and text.endswith("lds"):
            copies += 1
            used = set().union(*(_sgprs(w) for o in ops for w in o.split()))
            if m0 < 1 or any(since.get(r, 99) < 5 for r in used):
                bad.append((i, text))
        states = 1 + (int(ops[0], 0) if op == "s_nop" else 0)
        since = {r: n + states for r, n in since.items() if n + states < 8}
        m0 += states
        if op.startswith("v_"):
            since.update((r, 0) for r in _sgprs(ops[0].split()[0] if ops[0] else ""))
        if ops[0] == "m0":
            m0 = 0
    return copies, bad


def test_checker_finds_planted_hazards():
    ok = ["v_readfirstlane_b32 s4, v0", "s_nop 4", "s_add_u32 m0, s9, 0x400", "s_nop 0",
          "buffer_load_dwordx4 v6, s[4:7], s1 offen lds"]
    assert hazards(ok) == (1, [])
    assert len(hazards(ok[:1] + ok[2:])[1]) == 1  # the descriptor word is read 2 wait states after its VALU write
    assert len(hazards(ok[:3] + ok[4:])[1]) == 1  # M0 is read in the next state


def test_copies_keep_their_wait_states(tmp_path):
    if not os.path.exists(OBJDUMP):
        pytest.skip("llvm-objdump of the ROCm toolchain not found")
    lib = shutil.copy(_lib.LIB_PATH, tmp_path)
    subprocess.run([OBJDUMP, "--offloading", lib], cwd=tmp_path, check=True, capture_output=True)
    copies, bad = 0, []
    for f in sorted(os.listdir(tmp_path)):
        if "gfx950" in f:
            asm = subprocess.run([OBJDUMP, "-d", f], cwd=tmp_path, check=True, capture_output=True, text=True).stdout
            n, b = hazards(asm.splitlines())
            copies, bad = copies + n, bad + b
    assert copies > 1000, copies
    assert not bad, bad[:10]

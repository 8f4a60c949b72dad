"""Build-time check of the wait states that the inline-asm copies of the GEMM kernels rely on (csrc/gemm_common.h,
buf2lds_inner): no VALU instruction may write an SGPR operand (or M0) of a `buffer_load ... lds` in the five wait states
before it, and any write of M0 must be one wait state ahead.  The compiler tracks neither for inline asm, and whether its
code keeps them depends on its register allocation, so every build is checked and one that breaks a rule is refused."""
from __future__ import annotations

import os
import re
import shutil
import subprocess
import tempfile

VALU_SGPR_STATES = 5  # VALU write of an SGPR -> a VMEM instruction that reads it
M0_STATES = 1         # any write of M0 -> a copy to LDS

_INSN = re.compile(r"\s+([a-z]\w+)(?:\s+(.*?))?\s*//\s*([0-9A-Fa-f]+):")
_LABEL = re.compile(r"[0-9A-Fa-f]+ <(.+)>:\s*$")
_TARGET = re.compile(r"<.*>\s*$")
# VALU instructions with a second destination: a carry or a scale flag in SGPRs
_TWO_DST = re.compile(r"v_(\w*_co_|div_scale_|mad_u64_|mad_i64_)")
_ENDS = ("s_branch", "s_endpgm", "s_code_end", "s_setpc", "s_swappc")


def objdump() -> str:
    p = os.path.join(os.environ.get("ROCM_PATH", "/opt/rocm"), "llvm", "bin", "llvm-objdump")
    p = p if os.path.exists(p) else shutil.which("llvm-objdump")
    if p is None:
        raise RuntimeError("llvm-objdump of the ROCm toolchain not found: the wait states of the built copies cannot be checked")
    return p


def _sgprs(operand):
    m = re.match(r"s\[(\d+):(\d+)\]$", operand)
    if m:
        return {f"s{i}" for i in range(int(m[1]), int(m[2]) + 1)}
    if re.match(r"s\d+$", operand):
        return {operand}
    return {"vcc_lo", "vcc_hi"} if operand == "vcc" else {operand} if operand in ("m0", "vcc_lo", "vcc_hi") else set()


class _Insn:
    __slots__ = ("addr", "op", "ops", "text", "entry", "target")

    def __init__(self, addr, op, rest, text, entry, target):
        self.addr, self.op, self.text, self.entry, self.target = addr, op, text, entry, target
        self.ops = [o.strip() for o in rest.split(",")] if rest else []

    def states(self):
        return 1 + (int(self.ops[0], 0) if self.op == "s_nop" else 0)

    def written(self):
        """SGPRs a VALU instruction writes, and M0 of any instruction."""
        if not self.ops or self.op.startswith(("s_cbranch", "s_branch", "s_cmp", "s_bitcmp")):
            return set()
        dst = self.ops[:2] if _TWO_DST.match(self.op) else self.ops[:1]
        w = set().union(*(_sgprs(o.split()[0]) for o in dst if o))
        return w if self.op.startswith("v_") else w & {"m0"}


def _parse(lines):
    """Instructions of an llvm-objdump listing.  A branch's target is its address field plus 4 plus 4 times its signed
    16-bit offset."""
    out, entry = [], True
    for line in lines:
        if _LABEL.match(line):
            entry = True
            continue
        m = _INSN.match(line)
        if not m:
            continue
        op, rest, addr = m[1], m[2] or "", int(m[3], 16)
        target = None
        if op.startswith(("s_branch", "s_cbranch")):
            off = int(rest.split()[0], 0) & 0xffff
            target = addr + 4 + 4 * (off - 0x10000 if off & 0x8000 else off)
        out.append(_Insn(addr, op, rest, line.split("//")[0].strip(), entry, target))
        entry = False
    return out


def hazards(lines):
    """(copies seen, [(address, text)] of the copies that break a rule) of an llvm-objdump -d listing.  Every copy is
    followed backwards over all ways that lead to it (fall-through and branches, loops' back edges among them) as far as
    the rules reach."""
    insns = _parse(lines)
    at = {x.addr: i for i, x in enumerate(insns)}
    jumps = {}  # index -> indices of the branches that go there
    for i, x in enumerate(insns):
        if x.target is not None:
            if x.target not in at:
                raise RuntimeError(f"branch to an unknown address: {x.text}")
            jumps.setdefault(at[x.target], []).append(i)
        elif x.op.startswith(("s_setpc", "s_swappc", "s_cbranch_g", "s_cbranch_i", "s_call")):
            raise RuntimeError(f"indirect control flow cannot be followed: {x.text}")

    def preds(i):
        p = list(jumps.get(i, ()))
        if i > 0 and not insns[i].entry and not insns[i - 1].op.startswith(_ENDS):
            p.append(i - 1)
        return p

    copies, bad = 0, []
    for c, x in enumerate(insns):
        if not (x.op.startswith("buffer_load") and x.text.endswith("lds")):
            continue
        copies += 1
        used = {"m0"}.union(*(_sgprs(w) for o in x.ops for w in o.split()))
        nearest = {}  # index -> fewest wait states between it and the copy
        todo = [(p, 0) for p in preds(c)]
        while todo:
            i, n = todo.pop()
            if n >= VALU_SGPR_STATES or nearest.get(i, VALU_SGPR_STATES) <= n:
                continue
            nearest[i] = n
            hit = insns[i].written() & used
            if hit and (insns[i].op.startswith("v_") or n < M0_STATES):
                bad.append((x.addr, x.text))
                break
            todo += [(p, n + insns[i].states()) for p in preds(i)]
    return copies, bad


def check(lib: str):
    """hazards() of every GPU code object in a built library."""
    tool = objdump()
    copies, bad = 0, []
    with tempfile.TemporaryDirectory() as tmp:
        local = shutil.copy(lib, os.path.join(tmp, "lib.so"))
        subprocess.run([tool, "--offloading", local], cwd=tmp, check=True, capture_output=True)
        for f in sorted(os.listdir(tmp)):
            if "amdgcn" in f:
                asm = subprocess.run([tool, "-d", f], cwd=tmp, check=True, capture_output=True, text=True).stdout
                n, b = hazards(asm.splitlines())
                copies, bad = copies + n, bad + b
    return copies, bad

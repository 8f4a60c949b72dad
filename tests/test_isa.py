"""The wait states the inline-asm copies of the GEMM kernels rely on (csrc/gemm_common.h, buf2lds_inner): the checker that
every build runs (isa_check.py) finds planted violations, on a branch and a loop's back edge too, a build that has one is
refused, and the built library has none."""
import pytest

from trenowanie_generatora_obrazkow_amd import _lib, isa_check

COPY = "buffer_load_dwordx4 v6, s[4:7], s1 offen lds"


def _listing(lines):
    """llvm-objdump's form: 4-byte instructions from address 0x100 on; "label:" starts a function, and a branch names the
    index of the instruction it goes to."""
    out, n = [], 0
    insns = [t for t in lines if not t.endswith(":")]
    for t in lines:
        if t.endswith(":"):
            out.append(f"{0x100 + 4 * n:016x} <{t[:-1]}>:")
            continue
        op, _, rest = t.partition(" ")
        if op.startswith(("s_branch", "s_cbranch")):
            assert 0 <= int(rest) < len(insns)
            t = f"{op} {(int(rest) - n - 1) & 0xffff}"
        out.append(f"\t{t:<60}// {0x100 + 4 * n:012X}: 00000000")
        n += 1
    return out


def _bad(*lines):
    copies, bad = isa_check.hazards(_listing(lines))
    assert copies == sum(t.endswith("lds") for t in lines)
    return len(bad)


def test_checker_finds_planted_hazards():
    ok = ["f:", "v_readfirstlane_b32 s4, v0", "s_nop 4", "s_add_u32 m0, s9, 0x400", "s_nop 0", COPY, "s_endpgm"]
    assert _bad(*ok) == 0
    assert _bad(*ok[:2], *ok[3:]) == 1  # the descriptor word is read 2 wait states after its VALU write
    assert _bad(*ok[:4], *ok[5:]) == 1  # M0 is read in the next state
    assert _bad("f:", "v_readfirstlane_b32 s1, v0", "s_nop 3", COPY, "s_endpgm") == 1  # the offset, 4 states
    assert _bad("f:", "v_readfirstlane_b32 s8, v0", COPY, "s_endpgm") == 0  # a register the copy does not read


@pytest.mark.parametrize("write", ["v_add_co_u32_e64 v0, s[4:5], v1, v2", "v_mad_u64_u32 v[0:1], s[6:7], s3, v2, 0",
                                   "v_div_scale_f32 v0, s[0:1], v1, v2, v3", "v_readfirstlane_b32 m0, v0"])
def test_second_destinations_and_m0(write):
    assert _bad("f:", write, "s_nop 3", COPY, "s_endpgm") == 1
    assert _bad("f:", write, "s_nop 4", COPY, "s_endpgm") == 0


def test_checker_follows_control_flow():
    # a write at a loop's end is next to the copy at its head
    loop = ["f:", "s_nop 7", COPY, "s_nop 7", "v_readfirstlane_b32 s4, v0", "s_cbranch_scc1 1", "s_endpgm"]
    assert _bad(*loop) == 1
    assert _bad(*loop[:5], "s_nop 3", *loop[5:]) == 0  # 4 states of the nop and the branch's own
    # a write ahead of a branch over a long block
    skip = ["f:", "v_readfirstlane_b32 s5, v0", "s_cbranch_vccz 4", "s_nop 7", "s_nop 7", COPY, "s_endpgm"]
    assert _bad(*skip) == 1
    # no way leads past an unconditional branch or from another function's end
    assert _bad("f:", "s_branch 2", "v_readfirstlane_b32 s5, v0", COPY, "s_endpgm") == 1
    assert _bad("f:", "s_branch 3", "v_readfirstlane_b32 s5, v0", "s_endpgm", COPY, "s_endpgm") == 0
    assert _bad("f:", "v_readfirstlane_b32 s5, v0", "s_branch 0", COPY, "s_endpgm") == 0
    assert _bad("f:", "v_readfirstlane_b32 s5, v0", "g:", COPY, "s_endpgm") == 0
    with pytest.raises(RuntimeError):
        isa_check.hazards(_listing(["f:", "s_setpc_b64 s[0:1]", COPY, "s_endpgm"]))


def test_copies_keep_their_wait_states():
    copies, bad = isa_check.check(_lib.LIB_PATH)
    assert copies > 1000, copies
    assert not bad, bad[:10]


def test_build_refuses_a_hazard(monkeypatch, tmp_path):
    """build() installs nothing when the check finds a violation (the compiler's runs are left out)."""
    from trenowanie_generatora_obrazkow_amd import build as hb
    monkeypatch.setattr(hb, "LIB_DIR", str(tmp_path))
    monkeypatch.setattr(hb, "LIB", str(tmp_path / "lib.so"))

    class Done:
        returncode, stderr = 0, ""

    monkeypatch.setattr(hb.subprocess, "run", lambda cmd, **kw: (open(cmd[-1], "w").close(), Done())[1])
    monkeypatch.setattr(hb.isa_check, "check", lambda lib: (1, [(0x100, COPY)]))
    with pytest.raises(RuntimeError, match="wait state"):
        hb.build()
    assert not (tmp_path / "lib.so").exists()
    monkeypatch.setattr(hb.isa_check, "check", lambda lib: (1, []))
    assert hb.build() == str(tmp_path / "lib.so") and (tmp_path / "lib.so").exists()

"""What the compiler's listings say (CPU only).  Inline-assembly loads: what the check accepts, what it refuses, and that
the kernels as they are built here pass.  Log-prob forward: the loads that are meant to be in flight together are."""

import re

import pytest

from siirl_amd import asm_check, build

LOAD = [";;#ASMSTART", "global_load_dwordx4 v[4:7], v20, s[2:3]", ";;#ASMEND"]
DMA = [";;#ASMSTART", "s_mov_b32 m0, s4", "s_nop 0", "global_load_lds_dwordx4 v21, s[6:7]", ";;#ASMEND"]
WAIT = [";;#ASMSTART", "s_waitcnt vmcnt(0)", ";;#ASMEND"]
USE = ["v_mfma_f32_16x16x32_bf16 a[0:3], v[4:7], v[8:11], a[0:3]"]
END = ["s_endpgm"]


def _hazards(lines):
    text = "\n".join(["kernel:", *("\t" + x if not x.endswith(":") else x for x in lines), ".Lfunc_end0:"])
    return asm_check.check(text).get("kernel", [])


def test_accepts_what_is_waited_for():
    assert _hazards(LOAD + WAIT + USE + END) == []
    # one DMA after the load may stay in flight
    assert _hazards(LOAD + DMA + [";;#ASMSTART", "s_waitcnt vmcnt(1)", ";;#ASMEND"] + USE + END) == []
    # other registers may be used meanwhile; the compiler's own loads are its own business
    assert _hazards(LOAD + ["v_mov_b32_e32 v8, v9"] + WAIT + USE + END) == []
    assert _hazards(LOAD + WAIT + ["global_load_dwordx4 v[12:15], v20, s[2:3]", "v_mov_b32_e32 v1, v12"] + END) == []


@pytest.mark.parametrize("between", [
    ["v_mov_b32_e32 v30, v5"],  # copied before it arrives
    ["v_accvgpr_write_b32 a4, v7"],
    ["scratch_store_dwordx4 off, v[4:7], off offset:16"],  # spilled
    ["v_mov_b32_e32 v6, 0"],  # overwritten when it arrives
    ["v_add_u32_e32 v20, v4, v20"],
    LOAD,  # two loads into one place
    ["s_waitcnt lgkmcnt(0)"] + USE,  # the wrong counter
    [";;#ASMSTART", "s_waitcnt vmcnt(1)", ";;#ASMEND"] + USE,
])
def test_refuses_uses_before_the_wait(between):
    assert _hazards(LOAD + between + WAIT + USE + END)


def test_follows_branches_and_loops():
    # one side of a branch waits, the other does not
    assert _hazards(LOAD + ["s_cbranch_scc1 .LBB0_2"] + WAIT + [".LBB0_2:"] + USE + END)
    assert _hazards(LOAD + ["s_cbranch_scc1 .LBB0_2"] + WAIT + ["s_branch .LBB0_3", ".LBB0_2:"] + WAIT + [".LBB0_3:"] + USE +
                    END) == []
    # a load for the next pass, used at the head of the loop
    loop = [".LBB0_1:"] + USE + LOAD
    assert _hazards(LOAD + WAIT + loop + WAIT + ["s_cbranch_scc1 .LBB0_1"] + END) == []
    assert _hazards(LOAD + WAIT + loop + ["s_cbranch_scc1 .LBB0_1"] + WAIT + END)
    assert _hazards(LOAD + END) == ["s_endpgm with a load in flight"]


@pytest.fixture(scope="module")
def fused_linear():
    return build.listing(build.CSRC / "fused_linear.hip").read_text()


# the kernels whose inline-assembly loads fill registers: the ordinary GEMM and, for every A layout but the packed one, the one
# that reads W past the caches (those of gemm_short_k_kernel fill the LDS)
GEMMS = {"gemm_nt_kernel": 6, "gemm_once_kernel": 5}


def _gemms(names):
    return {g: sum(g in k for k in names) for g in GEMMS}


def test_the_kernels_as_built_pass(fused_linear):
    assert [s.name for s in build.sources() if build.has_asm_loads(s)] == ["fused_linear.hip"]
    assert _gemms(asm_check.kernels(fused_linear)) == GEMMS
    assert asm_check.check(fused_linear) == {}


def test_a_copy_in_the_real_kernel_is_seen(fused_linear):
    """The register that a step's first load fills, copied right behind the load: every one of those kernels is refused."""
    lines, out = fused_linear.splitlines(), []
    for line in lines:
        out.append(line)
        if "global_load_dwordx4 v[" in line and "offset:1024" in line:
            first = line.split("v[")[1].split(":")[0]
            out += [";;#ASMEND", f"\tv_mov_b32_e32 v0, v{first}", ";;#ASMSTART"]
    bad = asm_check.check("\n".join(out))
    assert _gemms(bad) == GEMMS


def test_log_prob_forward_waits_for_no_load_of_the_ragged_end_alone():
    """Every variant issues the ragged end's four loads together, waits for them and only then branches on what a lane has;
    with the ring, its sixteen loads go out together and the loop waits for the oldest four."""
    text = build.listing(build.CSRC / "logprob_entropy.hip").read_text()
    variants = {k: v for k, v in asm_check.kernels(text).items() if "lpe_fwd_kernel" in k}
    assert len(variants) == 24
    for name, body in variants.items():
        deep = re.search(r"Lb[01]ELb[01]ELb([01])E", name)[1] == "1"
        marks = "".join("L" if line.startswith("global_load_dwordx4") else "w" if "vmcnt" in line else "e" if "v_exp" in line
                        else "|" if line.endswith(":") or line.startswith(("s_branch", "s_cbranch")) else ""
                        for line, _ in body)
        if deep:
            assert "L" * 16 in marks and sum("vmcnt(12)" in line for line, _ in body) == 4, (name, marks)
        else:
            assert re.search(r"LLLLw+\|", marks), (name, marks)

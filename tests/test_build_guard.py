"""The build refuses kernels that spill registers (CPU only; nothing is compiled here).

Kernels that issue loads as inline assembly and wait for them by hand are only correct
while the compiler spills nothing; llaminar_amd.build parses the compiler's
kernel-resource-usage remarks and fails the build otherwise.
"""
import pytest

from llaminar_amd import build as b

REMARKS = """\
gemv_quad.h:702:1: remark: Function Name: _ZN6llamql16gemv_quad_kernelINS_7Q4KQuadELi1ELi{u}ELi0EEEvNS_8QuadArgsE [-Rpass-analysis=kernel-resource-usage]
  702 |     {{
      | ^
gemv_quad.h:702:1: remark:     TotalSGPRs: 48 [-Rpass-analysis=kernel-resource-usage]
gemv_quad.h:702:1: remark:     VGPRs: 128 [-Rpass-analysis=kernel-resource-usage]
gemv_quad.h:702:1: remark:     AGPRs: 0 [-Rpass-analysis=kernel-resource-usage]
gemv_quad.h:702:1: remark:     ScratchSize [bytes/lane]: {scratch} [-Rpass-analysis=kernel-resource-usage]
gemv_quad.h:702:1: remark:     Dynamic Stack: False [-Rpass-analysis=kernel-resource-usage]
gemv_quad.h:702:1: remark:     Occupancy [waves/SIMD]: 4 [-Rpass-analysis=kernel-resource-usage]
gemv_quad.h:702:1: remark:     SGPRs Spill: 0 [-Rpass-analysis=kernel-resource-usage]
gemv_quad.h:702:1: remark:     VGPRs Spill: {spill} [-Rpass-analysis=kernel-resource-usage]
gemv_quad.h:702:1: remark:     LDS Size [bytes/block]: 0 [-Rpass-analysis=kernel-resource-usage]
"""


def test_clean_kernels_pass_and_are_reported():
    text = REMARKS.format(u=3, scratch=0, spill=0) + REMARKS.format(u=2, scratch=0, spill=0)
    usage = b.check_kernel_resources(text, "gemv.hip")
    assert len(usage) == 2
    assert all(u["VGPRs"] == 128 and u["VGPRs Spill"] == 0 for u in usage.values())


@pytest.mark.parametrize("scratch,spill", [(60, 38), (4, 0), (0, 1)])
def test_a_spilling_kernel_fails_the_build(scratch, spill):
    text = REMARKS.format(u=3, scratch=0, spill=0) + REMARKS.format(u=4, scratch=scratch, spill=spill)
    with pytest.raises(b.SpillError) as e:
        b.check_kernel_resources(text, "gemv.hip")
    assert "Li4E" in str(e.value) and "Li3E" not in str(e.value)


# with -save-temps (which the build uses, for the assembly check below) the backend runs as a step of
# its own and prints the position AFTER "remark:", with column 0 and no source excerpt
REMARKS_SAVE_TEMPS = """\
remark: /root/repo/llaminar_amd/csrc/gemm.hip:195:0: Function Name: _ZN6llamql11gemm_kernelINS_9Q4KTraitsELb{d}EEEvNS_8GemmArgsE [-Rpass-analysis=kernel-resource-usage]
remark: /root/repo/llaminar_amd/csrc/gemm.hip:195:0:     TotalSGPRs: 68 [-Rpass-analysis=kernel-resource-usage]
remark: /root/repo/llaminar_amd/csrc/gemm.hip:195:0:     VGPRs: 128 [-Rpass-analysis=kernel-resource-usage]
remark: /root/repo/llaminar_amd/csrc/gemm.hip:195:0:     AGPRs: 0 [-Rpass-analysis=kernel-resource-usage]
remark: /root/repo/llaminar_amd/csrc/gemm.hip:195:0:     ScratchSize [bytes/lane]: {scratch} [-Rpass-analysis=kernel-resource-usage]
remark: /root/repo/llaminar_amd/csrc/gemm.hip:195:0:     Dynamic Stack: False [-Rpass-analysis=kernel-resource-usage]
remark: /root/repo/llaminar_amd/csrc/gemm.hip:195:0:     Occupancy [waves/SIMD]: 4 [-Rpass-analysis=kernel-resource-usage]
remark: /root/repo/llaminar_amd/csrc/gemm.hip:195:0:     SGPRs Spill: 0 [-Rpass-analysis=kernel-resource-usage]
remark: /root/repo/llaminar_amd/csrc/gemm.hip:195:0:     VGPRs Spill: {spill} [-Rpass-analysis=kernel-resource-usage]
remark: /root/repo/llaminar_amd/csrc/gemm.hip:195:0:     LDS Size [bytes/block]: 0 [-Rpass-analysis=kernel-resource-usage]
"""


def test_the_layout_of_the_remarks_under_save_temps_is_read_too():
    """A build that keeps the intermediate files prints 'remark: file:line:col: field', not 'file:line:col:
    remark: field'; a guard that only knew the second form let two spilling kernels through."""
    clean = REMARKS_SAVE_TEMPS.format(d=1, scratch=0, spill=0)
    usage = b.check_kernel_resources(clean, "gemm.hip")
    assert len(usage) == 1 and next(iter(usage.values()))["VGPRs"] == 128
    with pytest.raises(b.SpillError) as e:
        b.check_kernel_resources(clean + REMARKS_SAVE_TEMPS.format(d=0, scratch=44, spill=10), "gemm.hip")
    assert "Lb0E" in str(e.value) and "44 B/lane" in str(e.value) and "Lb1E" not in str(e.value)
    assert b._drop_resource_remarks(clean.splitlines()) == []


def test_remarks_do_not_reach_the_build_log():
    lines = (REMARKS.format(u=3, scratch=0, spill=0) + "x.hip:1:1: warning: something real\n").splitlines()
    assert b._drop_resource_remarks(lines) == ["x.hip:1:1: warning: something real"]


def test_compile_command_asks_for_the_remarks():
    assert b.RESOURCE_FLAG == "-Rpass-analysis=kernel-resource-usage"


def test_a_refused_object_is_not_kept(tmp_path, monkeypatch):
    """A build without force keeps objects newer than their sources: one that the checks refused must not be there."""
    source, stderr = tmp_path / "demo.hip", REMARKS.format(u=4, scratch=4, spill=0)
    source.write_text("")

    def compiler(cmd, **_):
        (tmp_path / "demo.o").write_text("object")
        return b.subprocess.CompletedProcess(cmd, 0, "", stderr)

    monkeypatch.setattr(b, "OBJDIR", tmp_path)
    monkeypatch.setattr(b, "_headers_mtime", lambda: 0.0)
    monkeypatch.setattr(b, "hipcc", lambda: "hipcc")
    monkeypatch.setattr(b.subprocess, "run", compiler)
    for _ in range(2):
        with pytest.raises(b.SpillError):
            b._compile(source, force=False)
    stderr = REMARKS.format(u=4, scratch=0, spill=0)
    assert b._compile(source, force=False).exists()


# ---- the second check: registers of hand-issued loads touched before their wait ----------

_PROLOGUE = """\
\t.text
_ZN6llamql4demoEv:
\ts_load_dwordx2 s[0:1], s[4:5], 0x0
"""


def _asm(body: str) -> str:
    return _PROLOGUE + body + "\ts_endpgm\n"


def test_inflight_check_accepts_use_after_wait():
    from llaminar_amd.build import check_inflight_registers

    asm = _asm("""\
\t;;#ASMSTART
\tglobal_load_dwordx4 v[8:11], v[2:3], off
\t;;#ASMEND
\t;;#ASMSTART
\tglobal_load_dwordx4 v[12:15], v[2:3], off offset:16
\t;;#ASMEND
\tv_add_u32_e32 v20, v21, v22
\t;;#ASMSTART
\ts_waitcnt vmcnt(1)
\t;;#ASMEND
\tv_and_b32_e32 v4, 0xf0f0f0f, v8
\t;;#ASMSTART
\ts_waitcnt vmcnt(0)
\t;;#ASMEND
\tv_and_b32_e32 v5, 0xf0f0f0f, v12
""")
    assert check_inflight_registers(asm, "demo.hip") == 2


def test_inflight_check_refuses_a_copy_before_the_wait():
    from llaminar_amd.build import InFlightRegisterError, check_inflight_registers

    asm = _asm("""\
\t;;#ASMSTART
\tglobal_load_dwordx4 v[8:11], v[2:3], off
\t;;#ASMEND
\tv_mov_b64_e32 v[20:21], v[8:9]
\t;;#ASMSTART
\ts_waitcnt vmcnt(0)
\t;;#ASMEND
""")
    with pytest.raises(InFlightRegisterError, match="v8"):
        check_inflight_registers(asm, "demo.hip")


def test_inflight_check_refuses_partial_wait_and_reuse_as_address():
    from llaminar_amd.build import InFlightRegisterError, check_inflight_registers

    # vmcnt(1) retires the older load only: the newer one's registers are still in flight
    asm = _asm("""\
\t;;#ASMSTART
\tglobal_load_dwordx4 v[8:11], v[2:3], off
\t;;#ASMEND
\t;;#ASMSTART
\tglobal_load_dwordx2 v[12:13], v[2:3], off offset:16
\t;;#ASMEND
\t;;#ASMSTART
\ts_waitcnt vmcnt(1)
\t;;#ASMEND
\tv_add_u32_e32 v4, v8, v12
""")
    with pytest.raises(InFlightRegisterError, match="v12"):
        check_inflight_registers(asm, "demo.hip")
    # the destination of a load in flight handed out as an address of the next load
    asm = _asm("""\
\t;;#ASMSTART
\tglobal_load_dwordx2 v[8:9], v[2:3], off
\t;;#ASMEND
\t;;#ASMSTART
\tglobal_load_dwordx4 v[16:19], v[8:9], off
\t;;#ASMEND
""")
    with pytest.raises(InFlightRegisterError, match="in flight"):
        check_inflight_registers(asm, "demo.hip")


def test_inflight_check_counts_other_memory_operations_and_resets_at_jumps():
    from llaminar_amd.build import check_inflight_registers

    # a compiler-issued store after the load is one more entry of vmcnt: vmcnt(1) then means
    # "the hand-issued load has landed"; after an unconditional branch nothing is assumed in flight
    asm = _asm("""\
\t;;#ASMSTART
\tglobal_load_dwordx4 v[8:11], v[2:3], off
\t;;#ASMEND
\tglobal_store_dword v[30:31], v32, off
\t;;#ASMSTART
\ts_waitcnt vmcnt(1)
\t;;#ASMEND
\tv_mov_b32_e32 v4, v8
\t;;#ASMSTART
\tglobal_load_dwordx4 v[12:15], v[2:3], off
\t;;#ASMEND
\ts_branch .LBB0_2
.LBB0_1:
\tv_mov_b32_e32 v5, v12
.LBB0_2:
\ts_waitcnt vmcnt(0)
""")
    assert check_inflight_registers(asm, "demo.hip") == 2


LOOP = """\
\t;;#ASMSTART
\tglobal_load_dwordx4 v[8:11], v[2:3], off
\t;;#ASMEND
.LBB0_1:
\t;;#ASMSTART
\ts_waitcnt vmcnt(0)
\t;;#ASMEND
\tv_and_b32_e32 v4, 0xf0f0f0f, v{read}
\t;;#ASMSTART
\tglobal_load_dwordx4 v[{dst}], v[2:3], off
\t;;#ASMEND
\t{between}
\ts_cbranch_scc1 .LBB0_1
\ts_waitcnt vmcnt(0)
"""


def test_inflight_check_follows_a_loop_edge():
    from llaminar_amd.build import InFlightRegisterError, check_inflight_registers

    assert check_inflight_registers(_asm(LOOP.format(read=8, dst="8:11", between="s_nop 0")), "demo.hip") == 2
    # the next turn's load lands in other registers, and a copy that brings them to where the loop begins is taken on the
    # edge, ahead of the wait behind the label: in program order the copy comes before the load
    edge = LOOP.format(read=8, dst="12:15", between="s_branch .LBB0_3").replace(
        ".LBB0_1:", "\ts_branch .LBB0_1\n.LBB0_2:\n\tv_mov_b64_e32 v[8:9], v[12:13]\n.LBB0_1:") + \
        ".LBB0_3:\n\ts_cbranch_scc1 .LBB0_2\n\ts_waitcnt vmcnt(0)\n"
    with pytest.raises(InFlightRegisterError, match="v12"):
        check_inflight_registers(_asm(edge), "demo.hip")
    with pytest.raises(InFlightRegisterError, match="v8"):   # behind a conditional jump over the wait
        check_inflight_registers(_asm("""\
\t;;#ASMSTART
\tglobal_load_dwordx4 v[8:11], v[2:3], off
\t;;#ASMEND
\ts_cbranch_vccz .LBB0_2
\ts_waitcnt vmcnt(0)
.LBB0_2:
\tv_mov_b32_e32 v4, v8
"""), "demo.hip")


# ---- scalar registers that a vector instruction has just written ---------------------------------

SCALAR = """\
_Z6kernelv:
\tv_readfirstlane_b32 s7, v3
{between}
\t;;#ASMSTART
\tglobal_load_dwordx4 v[18:21], v2, s[6:7] offset:16
\t;;#ASMEND
\ts_endpgm
"""


@pytest.mark.parametrize("between", ["", "\ts_nop 3", "\tv_mov_b32_e32 v1, v2\n\ts_nop 2", "\tv_mul_u32_u24_e32 v3, 0x90, v4\n.LBB0_1:\n\ts_nop 0"])
def test_a_load_too_soon_after_its_base_was_made_fails_the_build(between):
    with pytest.raises(b.ScalarHazardError, match="s7"):
        b.check_scalar_hazards(SCALAR.format(between=between), "moe.hip")


@pytest.mark.parametrize("between", ["\ts_nop 4", "\tv_mov_b32_e32 v1, v2\n\ts_nop 3", "\n".join(["\tv_mov_b32_e32 v1, v2"] * 5)])
def test_a_load_after_five_wait_states_passes(between):
    assert b.check_scalar_hazards(SCALAR.format(between=between), "moe.hip") == 1


def test_scalar_instructions_and_the_compilers_own_loads_need_no_wait():
    asm = SCALAR.format(between="").replace("v_readfirstlane_b32 s7, v3", "s_mov_b32 s7, s3")
    assert b.check_scalar_hazards(asm, "moe.hip") == 1
    own = SCALAR.format(between="").replace("\t;;#ASMSTART\n", "").replace("\t;;#ASMEND\n", "")
    assert b.check_scalar_hazards(own, "moe.hip") == 0


def test_the_wait_for_a_base_is_followed_over_jumps():
    loop = """\
_Z6kernelv:
.LBB0_1:
\t;;#ASMSTART
\tglobal_load_dwordx4 v[18:21], v2, s[6:7]
\t;;#ASMEND
\tv_readfirstlane_b32 s6, v3
{between}
\ts_cbranch_scc1 .LBB0_1
\ts_endpgm
"""
    with pytest.raises(b.ScalarHazardError, match="s6 4 wait states"):
        b.check_scalar_hazards(loop.format(between="\ts_nop 2"), "moe.hip")
    assert b.check_scalar_hazards(loop.format(between="\ts_nop 3"), "moe.hip") == 1
    # ahead of an unconditional jump, and what stands behind it in the text only
    with pytest.raises(b.ScalarHazardError, match="s6"):
        b.check_scalar_hazards(loop.format(between="\ts_branch .LBB0_1"), "moe.hip")
    past = "_Z6kernelv:\n\tv_readfirstlane_b32 s7, v3\n\ts_branch .LBB0_2\n.LBB0_1:\n" + SCALAR.split("{between}\n")[1] + ".LBB0_2:\n\ts_endpgm\n"
    assert b.check_scalar_hazards(past, "moe.hip") == 1


# ---- m0, just before a load into LDS -----------------------------------------------------------------

TO_LDS = """\
_Z6kernelv:
\t;;#ASMSTART
\ts_mov_b32 m0, s5
{between}
\t{load}
\t;;#ASMEND
\ts_endpgm
"""
LDS_LOADS = ["global_load_lds_dwordx4 v2, s[6:7]", "global_load_lds_dword v[2:3], off", "buffer_load_dword v2, s[8:11], 0 offen lds"]


@pytest.mark.parametrize("load", LDS_LOADS)
def test_a_load_into_lds_right_after_its_address_fails_the_build(load):
    for between in ("", "\t;;#ASMEND\n.LBB0_1:\n\t;;#ASMSTART"):
        with pytest.raises(b.ScalarHazardError, match="m0 0 wait states"):
            b.check_scalar_hazards(TO_LDS.format(between=between, load=load), "gemm.hip")
    for between in ("\ts_nop 0", "\ts_mov_b64 exec, s[2:3]"):
        assert b.check_scalar_hazards(TO_LDS.format(between=between, load=load), "gemm.hip") == 1


def test_loads_into_registers_need_no_wait_after_m0():
    assert b.check_scalar_hazards(TO_LDS.format(between="", load="global_load_dwordx4 v[8:11], v2, s[6:7]"), "gemm.hip") == 1

"""The build refuses kernels that keep loads in flight and spill registers (qwen-llm_amd/build.py): the check on
hipcc's resource-usage remarks, fed with remark text of the shape the compiler prints; and code that touches a register
ahead of its load's wait (qwen-llm_amd/inflight.py), fed with short kernels.  Host logic, no GPU."""
import importlib.util
import os

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def _build_module(name="build"):
    spec = importlib.util.spec_from_file_location(f"_dflash_{name}_for_test", os.path.join(ROOT, "qwen-llm_amd", name + ".py"))
    mod = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(mod)
    return mod


def remarks(name, vgpr_spill, scratch=0):
    tag = "[-Rpass-analysis=kernel-resource-usage]"
    lines = [f"x.hip:10:1: remark: Function Name: {name} {tag}", "   10 | __global__ void k() {", "      | ^"]
    for key, val in (("TotalSGPRs", 100), ("VGPRs", 120), ("ScratchSize [bytes/lane]", scratch), ("VGPRs Spill", vgpr_spill)):
        lines += [f"x.hip:10:1: remark:     {key}: {val} {tag}", "   10 | __global__ void k() {", "      | ^"]
    return "\n".join(lines) + "\n"


def test_a_guarded_kernel_that_spills_is_refused():
    b = _build_module()
    bad = b.check_no_scratch(remarks("_ZN12_GLOBAL__N_123gemm_q4k_experts_kernelIffLb0EEEvPKh", 13, 52), expect=())
    assert len(bad) == 2 and all("gemm_q4k_experts_kernel" in m for m in bad) and "52" in bad[0] and "13" in bad[1]
    # a scratch frame without a spill count is refused as well
    bad = b.check_no_scratch(remarks("_ZN12_GLOBAL__N_123gemm_q4k_experts_kernelIffLb0EEEvPKh", 0, 16), expect=())
    assert len(bad) == 1 and "scratch" in bad[0]


def test_remarks_with_their_place_behind_the_word_are_read_too():
    b = _build_module()
    name = "_ZN12_GLOBAL__N_123gemm_q4k_experts_kernelIffLb0EEEvPKh"
    for spills, scratch, complaints in ((0, 0, 0), (13, 52, 2)):
        lines = [line.replace("x.hip:10:1: remark: ", "remark: x.hip:10:0: ") for line in remarks(name, spills, scratch).splitlines() if "remark" in line]
        assert len(b.check_no_scratch("\n".join(lines), expect=("gemm_q4k_experts_kernel",))) == complaints
        assert b.strip_remarks("\n".join(lines + ["y.hip:3:5: warning: w"])) == "y.hip:3:5: warning: w"


def test_guarded_kernels_without_spills_and_other_kernels_pass():
    b = _build_module()
    text = remarks("_ZN12_GLOBAL__N_121gemm_q4k_tiled_kernelIfEEvPKh", 0) + remarks("_Z15rms_norm_kernelPKf", 7, 28)
    assert b.check_no_scratch(text, expect=()) == []


def test_a_guarded_kernel_missing_from_the_remarks_fails_the_guard():
    """A changed remark format or a dropped flag must not make the guard pass vacuously."""
    b = _build_module()
    text = remarks("_ZN12_GLOBAL__N_121gemm_q4k_tiled_kernelIfEEvPKh", 0)
    bad = b.check_no_scratch(text)  # every other guarded kernel is unreported
    assert len(bad) == len(b.NO_SCRATCH_KERNELS) - 1 and all("no resource-usage remark" in m for m in bad)
    assert b.check_no_scratch("nothing of the kind\n", expect=("gemm_q4k_tiled_kernel",)) != []


def test_every_kernel_that_waits_for_memory_by_hand_is_guarded():
    """A kernel with an s_waitcnt of its own on vector memory, or a call of a function that waits, is named in the build's list, and a
    file that such a kernel lives in has its generated code checked."""
    import re

    b = _build_module()
    found = set()
    for src in b.sources():
        with open(src) as f:
            text = re.sub(r"//[^\n]*", "", f.read())
        name = os.path.basename(src)
        for at in [m.end() for m in re.finditer("__global__", text)]:
            kernel = re.compile(r"(\w+_kernel)\s*\(").search(text, at)
            body = text[kernel.end():text.index("\n}\n", at)]
            # (a wait for LDS alone, or for everything, is none of this)
            if re.search(r"__builtin_amdgcn_s_waitcnt\((?!kWaitLds\)|0\)|0xC07F\))|\b\w*wait_(?:vm\w*|groups)\(|\b(?:wide|attn)_wait\(", body):
                found.add(kernel.group(1))
                assert kernel.group(1) in b.NO_SCRATCH_BY_FILE.get(name, ()), f"{name}: {kernel.group(1)}"
                assert name in b.CHECKED_CODE, name
    assert len(found) >= 8


def test_inspected_exceptions_hold_only_at_their_recorded_counts():
    b = _build_module()
    b.INSPECTED_SPILLS = {"gemm_q6k_stream_kernelILi16EfE": 13}
    name = "_ZN12_GLOBAL__N_122gemm_q6k_stream_kernelILi16EfEEvPKhPKT0_PfS6_iiii"
    assert b.check_no_scratch(remarks(name, 13), expect=()) == []
    assert len(b.check_no_scratch(remarks(name, 14), expect=())) == 1
    assert len(b.check_no_scratch(remarks(name, 0), expect=())) == 1  # the code changed: read the generated code again


def test_remarks_are_stripped_from_what_the_build_prints():
    b = _build_module()
    text = remarks("_Z1kv", 0) + "y.hip:3:5: warning: unused variable 'q' [-Wunused-variable]\n    3 |     int q;\n"
    out = b.strip_remarks(text)
    assert "remark" not in out and "unused variable 'q'" in out


def kernel(*code, name="k"):
    return "\n".join([f"{name}:                  ; @{name}", *code, "\ts_endpgm", "\t.section\t.rodata", f"\t.amdhsa_kernel {name}",
                      "\t.end_amdhsa_kernel", "\t.text", ".Lfunc_end0:"]) + "\n"


READS = ["\tds_read_b128 v[4:7], v0", "\tds_read_b128 v[8:11], v0 offset:16", "\tds_read_u16 v12, v1"]


@pytest.mark.parametrize("code", [
    READS + ["\ts_waitcnt lgkmcnt(2)", "\tv_mov_b32_e32 v20, v7", "\ts_waitcnt lgkmcnt(1)", "\tv_mfma_f32_16x16x32_f16 a[0:3], v[4:7], v[8:11], a[0:3]"],
    # a wait for another counter in between, copies into LDS and a store, which are not later reads
    READS + ["\tglobal_load_lds_dwordx4 v[30:31], off", "\tds_write_b32 v1, v2", "\ts_waitcnt lgkmcnt(0)", "\tv_mov_b32_e32 v8, v12"],
    # both ways of a branch wait; the other counter's loads are not followed unless asked for
    READS + ["\ts_cbranch_scc0 .LBB0_2", "\ts_waitcnt lgkmcnt(0)", "\ts_branch .LBB0_3", ".LBB0_2:", "\ts_waitcnt vmcnt(3) lgkmcnt(0)", ".LBB0_3:",
             "\tv_mov_b32_e32 v20, v7", "\tglobal_load_dword v3, v[4:5], off", "\tv_mov_b32_e32 v6, v3"],
])
def test_registers_touched_behind_their_wait_pass(code):
    assert _build_module("inflight").check_assembly(kernel(*code)) == []


@pytest.mark.parametrize("code,register", [
    (READS + ["\tv_mov_b32_e32 v20, v7"], "v7"),  # the copy that a register allocator may make
    (READS + ["\ts_waitcnt lgkmcnt(2)", "\tv_mov_b32_e32 v20, v8"], "v8"),  # one read too few waited for
    (READS + ["\ts_waitcnt vmcnt(0)", "\tv_mov_b32_e32 v20, v12"], "v12"),  # the wrong counter
    (READS + ["\tv_mov_b32_e32 v9, 0", "\ts_waitcnt lgkmcnt(0)"], "v9"),  # written ahead of the arrival
    (["\tds_read_b128 a[4:7], v0", "\tv_accvgpr_read_b32 v1, a5"], "a5"),
    (READS[:1] + ["\tds_write_b32 v1, v2", "\ts_waitcnt lgkmcnt(1)", "\tv_mov_b32_e32 v20, v4"], "v4"),  # (only reads count)
    # one way of a branch does not wait; a read at a loop's end, touched at its head
    (READS + ["\ts_cbranch_scc0 .LBB0_2", "\ts_waitcnt lgkmcnt(0)", ".LBB0_2:", "\tv_mov_b32_e32 v20, v7"], "v7"),
    ([".LBB0_1:", "\tv_mov_b32_e32 v20, v4", "\ts_waitcnt lgkmcnt(0)", "\tds_read_b32 v4, v0", "\ts_cbranch_scc1 .LBB0_1"], "v4"),
])
def test_registers_touched_ahead_of_their_wait_are_refused(code, register):
    bad = _build_module("inflight").check_assembly(kernel(*code))
    assert len(bad) == 1 and register in bad[0] and "in flight" in bad[0]


def test_loads_from_memory_are_followed_where_asked_for_and_named_kernels_must_be_there():
    m = _build_module("inflight")
    code = ["\tglobal_load_dwordx4 v[4:7], v0, s[2:3]", "\tglobal_load_lds_dwordx4 v[8:9], off", "\ts_waitcnt vmcnt(1)", "\tv_mov_b32_e32 v1, v4"]
    assert m.check_assembly(kernel(*code), memory=("k",)) == []
    code[2] = "\ts_waitcnt vmcnt(2)"
    assert len(m.check_assembly(kernel(*code), memory=("k",))) == 1 and m.check_assembly(kernel(*code)) == []
    assert len(m.check_assembly(kernel(), memory=("gemm_rows_kernel",))) == 1


def test_a_file_without_its_assembly_is_refused(tmp_path):
    assert len(_build_module().check_code("/x/gemm_rows.hip", str(tmp_path))) == 1

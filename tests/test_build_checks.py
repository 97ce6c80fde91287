"""Host-side checks of the build helpers (no GPU, no compiler run)."""

import time
from pathlib import Path

import pytest

from cornserve_amd import build
from cornserve_amd.build import check_hand_managed_acc_registers

_CLEAN = """
_Z6kernelv:
	v_add_u32_e32 v1, v2, v3
	;;#ASMSTART
	v_mfma_f32_16x16x32_bf16 a[0:3], v[0:3], v[4:7], a[0:3]
	;;#ASMEND
	ds_read_b128 v[8:11], v12
	;;#ASMSTART
	v_accvgpr_read_b32 v5, a[7]
	;;#ASMEND
	s_endpgm
"""

_SPILL = _CLEAN.replace("\tds_read_b128 v[8:11], v12\n", "\tv_accvgpr_write_b32 a17, v5\n\tds_read_b128 v[8:11], v12\n")
_STAGED = _CLEAN.replace("\tds_read_b128 v[8:11], v12\n", "\tglobal_load_dwordx4 a[0:3], v172, s[8:9] offset:256\n")
_COMPILER_ONLY = """
_Z7kernel2v:
	v_mfma_f32_16x16x32_bf16 a[0:3], v[0:3], v[4:7], a[0:3]
	v_accvgpr_read_b32 v5, a1
	s_endpgm
"""


def test_clean_kernel_passes():
    assert check_hand_managed_acc_registers(_CLEAN) == []


def test_compiler_spill_into_accumulation_register_is_reported():
    out = check_hand_managed_acc_registers(_SPILL)
    assert len(out) == 1 and out[0].startswith("_Z6kernelv")


def test_compiler_load_into_accumulation_register_is_reported():
    assert len(check_hand_managed_acc_registers(_STAGED)) == 1


def test_kernels_without_inline_accumulators_are_not_checked():
    # a kernel whose accumulators the compiler manages itself may use the registers freely
    assert check_hand_managed_acc_registers(_COMPILER_ONLY) == []
    assert len(check_hand_managed_acc_registers(_COMPILER_ONLY + _SPILL)) == 1


def test_an_object_whose_source_fails_the_check_does_not_survive(tmp_path, monkeypatch):
    """Compilation and check of a source run side by side: whichever ends first, an incremental build that follows a failed
    check must compile and check the source again instead of linking its object."""
    csrc, out = tmp_path / "csrc", tmp_path / "build"
    csrc.mkdir()
    (csrc / "a.hip").write_text(f"// {build.HAND_MANAGED_ACC_MARKER}\n")
    (csrc / "a.h").write_text("")
    linked = []

    def run(cmd):
        target = Path(cmd[cmd.index("-o") + 1])
        if "-shared" in cmd:
            linked.append(target)
        elif "-S" in cmd:
            target.write_text(_SPILL)
        else:
            time.sleep(0.3)        # the compilation outlasts the check
            target.write_text("object")

    monkeypatch.setattr(build, "CSRC", csrc)
    monkeypatch.setattr(build, "OBJ_DIR", out)
    monkeypatch.setattr(build, "_hipcc", lambda: "hipcc")
    monkeypatch.setattr(build, "_run", run)
    for force in (True, False):
        with pytest.raises(RuntimeError, match="accumulation registers"):
            build.build_library(force=force)
        assert not (out / "a.o").exists() and not linked


@pytest.mark.parametrize("listing,passes", [(_CLEAN, True), (_SPILL, False)])
def test_the_check_reads_the_listing_of_the_compilation_itself(tmp_path, monkeypatch, listing, passes):
    """One compilation gives object and listing; the object appears when the listing has passed, and nothing else stays."""
    commands = []

    def run(cmd):
        commands.append(cmd)
        target = Path(cmd[cmd.index("-o") + 1])
        target.write_text("object")
        (target.parent / f"a-hip-amdgcn-amd-amdhsa-{build.ARCH}.s").write_text(listing)

    monkeypatch.setattr(build, "OBJ_DIR", tmp_path)
    monkeypatch.setattr(build, "_run", run)
    obj = tmp_path / "a.o"
    if passes:
        build._compile_checked("hipcc", tmp_path / "a.hip", obj)
    else:
        with pytest.raises(RuntimeError, match="accumulation registers"):
            build._compile_checked("hipcc", tmp_path / "a.hip", obj)
    assert obj.exists() == passes and len(commands) == 1 and "-save-temps=obj" in commands[0]
    assert [p.name for p in tmp_path.iterdir()] == ["a.o"] * passes

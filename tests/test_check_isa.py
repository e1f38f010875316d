"""CPU check of fast-rbd-gradients_amd/check_isa.py, which the Makefile runs on
every library it links (any robot's): the samples are what the compiler has
produced, and the two libraries built here are clean."""
import os
import subprocess

import pytest

import check_isa
import common

JUMPED_OVER = """
<_Zkernel>:
\ts_and_saveexec_b64 s[0:1], vcc
\ts_cbranch_execz L0
\tv_add_f32_e32 v0, v1, v2
<L0>:
\ts_mov_b64 s[20:21], vcc
\tv_writelane_b32 v255, s20, 8
SAVE\tv_writelane_b32 v255, s21, 9
\ts_or_b64 exec, exec, s[0:1]
AFTER\tv_add_f32_e32 v0, v1, v2
"""
SHORT_BODY = """
<_Zkernel>:
\ts_and_saveexec_b64 s[0:1], vcc
\tv_add_f32_e32 v0, v1, v2
\ts_mov_b64 s[20:21], vcc
SAVE\tv_writelane_b32 v255, s21, 9
\ts_or_b64 exec, exec, s[0:1]
AFTER\tv_add_f32_e32 v0, v1, v2
"""
LOOP_EXIT = """
<_Zkernel>:
<L1>:
\tv_add_f32_e32 v0, v1, v2
\ts_andn2_b64 exec, exec, s[2:3]
\ts_cbranch_execnz L1
SAVE\ts_or_b64 exec, exec, s[0:1]
AFTER\tv_add_f32_e32 v0, v1, v2
"""
SAVES = ("v_accvgpr_write_b32 a2, v62", "scratch_store_dwordx2 off, v[110:111], off offset:4")


@pytest.mark.parametrize("save", SAVES)
@pytest.mark.parametrize("sample", [JUMPED_OVER, SHORT_BODY, LOOP_EXIT], ids=["jumped_over", "short_body", "loop_exit"])
def test_a_save_ahead_of_the_restore(sample, save):
    bad = sample.replace("SAVE", f"\t{save}\n").replace("AFTER", "")
    good = sample.replace("SAVE", "").replace("AFTER", f"\t{save}\n")
    assert {e[2] for e in check_isa.early_vector_writes(bad)} == {save}
    assert check_isa.early_vector_writes(good) == []


def test_a_bodys_own_last_instructions_are_not_it():
    asm = SHORT_BODY.replace("SAVE", "").replace("AFTER", "").replace(
        "\ts_mov_b64 s[20:21], vcc\n", "\ts_mov_b64 s[20:21], vcc\n\tv_mul_f32_e32 v3, v0, v0\n\tv_accvgpr_write_b32 a2, v3\n")
    assert check_isa.early_vector_writes(asm) == []


@pytest.mark.parametrize("lib", ["librbdgrad.so", "librbdgrad_arm7.so"])
def test_built_libraries_are_clean(lib):
    kernels, found = check_isa.check(os.path.join(common.PKG, lib))
    assert kernels > 150
    assert not found, found[:5]


def test_every_link_is_checked():
    for model in ([], ["MODEL=other", "URDF=other.urdf"]):
        r = subprocess.run(["make", "-n", "-B", "-C", common.PKG, *model, "-o", "other.urdf"],
                           capture_output=True, text=True)
        links = [ln for ln in r.stdout.replace("\\\n", " ").splitlines() if "-shared" in ln]
        assert len(links) == 1 and "check_isa.py" in links[0], r.stdout + r.stderr

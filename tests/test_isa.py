"""CPU check of the built libraries' gfx950 code: where lanes that sat out one
side of a branch are turned back on, no vector register may have been written
or saved before the instruction that turns them on.

The compiler can get this wrong when it runs out of scalar registers: it then
saves vector registers (to accumulation registers or scratch) at the start of
such a block, ahead of the instruction that restores the execution mask, so
the lanes that are still off save nothing and read garbage back.  It did so in
FP64-column kernels: wrong gradients, and stores to garbage addresses."""
import os
import re
import subprocess

import pytest

import common

OBJDUMP = "/opt/rocm/llvm/bin/llvm-objdump"
RESTORE = re.compile(r"s_(or|andn2|xor)_b64 exec,|s_or_saveexec_b64|s_andn2_saveexec_b64")
END = re.compile(r"s_cbranch|s_branch|s_endpgm|s_and_saveexec_b64|s_setpc|s_swappc")
HARMLESS = ("v_writelane", "v_readlane", "v_readfirstlane", "v_cmp")     # scalar results, or into spilled scalars


def early_vector_writes(asm):
    """[(function, label, instruction)] of vector instructions between the
    label of a block that an s_cbranch_execz jumps to and the instruction that
    restores the execution mask there."""
    found = []
    for part in re.split(r"\n(?=<_Z)", asm):
        name = part.split(">", 1)[0].lstrip("<\n")
        lines = [ln.split("//")[0].strip() for ln in part.splitlines()[1:]]
        targets = set(re.findall(r"s_cbranch_execz (\w+)", part))
        at = {m.group(1): i for i, ln in enumerate(lines) if (m := re.match(r"<(\w+)>:$", ln))}
        for label in targets & set(at):
            early = []
            for ln in lines[at[label] + 1:]:
                if re.match(r"<\w+>:$", ln) or END.match(ln):
                    break
                if RESTORE.match(ln):
                    found += [(name, label, e) for e in early]
                    break
                if ln.startswith(("v_", "ds_", "global_", "scratch_", "buffer_", "flat_")) and \
                        not ln.startswith(HARMLESS):
                    early.append(ln)
    return found


def test_the_scan_sees_a_save_ahead_of_the_restore():
    bad = """
<_Zkernel>:
\ts_and_saveexec_b64 s[0:1], vcc
\ts_cbranch_execz L0
\tv_add_f32_e32 v0, v1, v2
<L0>:
\tv_writelane_b32 v255, s46, 29
\tv_accvgpr_write_b32 a2, v62
\ts_or_b64 exec, exec, s[0:1]
\tv_add_f32_e32 v0, v1, v2
"""
    assert early_vector_writes(bad) == [("_Zkernel", "L0", "v_accvgpr_write_b32 a2, v62")]
    good = bad.replace("\tv_accvgpr_write_b32 a2, v62\n\ts_or_b64 exec, exec, s[0:1]\n",
                       "\ts_or_b64 exec, exec, s[0:1]\n\tv_accvgpr_write_b32 a2, v62\n")
    assert early_vector_writes(good) == []


@pytest.mark.parametrize("lib", ["librbdgrad.so", "librbdgrad_arm7.so"])
def test_no_vector_write_before_lanes_are_back(lib, tmp_path):
    path = os.path.join(common.PKG, lib)
    if not os.path.exists(path):
        pytest.skip(f"{lib} is not built")
    if not os.path.exists(OBJDUMP):
        pytest.skip("no llvm-objdump")
    os.symlink(path, tmp_path / lib)
    subprocess.run([OBJDUMP, "--offloading", lib], cwd=tmp_path, check=True, capture_output=True)
    objects = sorted(p for p in os.listdir(tmp_path) if p.endswith("gfx950"))
    assert len(objects) == 2, objects          # the flat and the batch kernels
    kernels, found = 0, []
    for obj in objects:
        asm = subprocess.run([OBJDUMP, "-d", "--symbolize-operands", "--no-show-raw-insn", "--no-leading-addr", obj],
                             cwd=tmp_path, check=True, capture_output=True, text=True).stdout
        kernels += asm.count("\n<_Z")
        found += early_vector_writes(asm)
    assert kernels > 150
    assert not found, found[:5]

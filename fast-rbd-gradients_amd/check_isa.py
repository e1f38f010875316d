#!/usr/bin/env python3
"""Checks a built library's gfx950 code for lanes that are turned back on too late.

    check_isa.py librbdgrad.so [...]      exit status 1 if a library holds a fault

After a divergent branch the code first restores the execution mask and only
then goes on with all lanes.  Short of scalar registers, the compiler may save
a vector register (to an accumulation register or scratch) at the start of
such a block but ahead of the restore: lanes that are still off save nothing
and read garbage back, values or addresses.  It depends on register pressure,
so a robot's tables or a small edit can bring it about in one kernel of many,
and tests may pass all the same; the Makefile therefore runs this on every
library it links, whichever robot it is for.

Looked at, for every kernel:
  * the block that s_cbranch_execz jumps to, up to the restore;
  * the code behind s_cbranch_execnz (a divergent loop's exit, all lanes off),
    up to the restore;
  * where a short body is not jumped over, what stands right before the
    restore: a save behind a copy or spill of scalar registers, the mark of
    this fault (a body's own last instructions are not).
"""
import os
import re
import subprocess
import sys
import tempfile

OBJDUMP = os.environ.get("LLVM_OBJDUMP", "/opt/rocm/llvm/bin/llvm-objdump")
RESTORE = re.compile(r"s_(or|andn2|xor)_b64 exec,|s_or_saveexec_b64|s_andn2_saveexec_b64")
END = re.compile(r"s_cbranch|s_branch|s_endpgm|s_and_saveexec_b64|s_setpc|s_swappc")
JOIN = re.compile(r"s_or_b64 exec, exec,|s_or_saveexec_b64 \S+, s")     # turns lanes back on without a branch's target
LABEL = re.compile(r"<(\w+)>:$")
VECTOR = ("v_", "ds_", "global_", "scratch_", "buffer_", "flat_")
HARMLESS = ("v_writelane", "v_readlane", "v_readfirstlane", "v_cmp")     # scalar results, or into spilled scalars
SAVE = re.compile(r"v_accvgpr_write_b32 a\d+, v\d+|scratch_store")
SCALAR_COPY = re.compile(r"s_mov_b(32|64) (s|vcc)|v_writelane_b32|v_readlane_b32")
WAIT = re.compile(r"s_nop|s_waitcnt")


def early_vector_writes(asm):
    """[(function, place, instruction)] of vector instructions ahead of the
    instruction that restores the execution mask, in llvm-objdump's text."""
    found = []
    for part in re.split(r"\n(?=<_Z)", asm):
        name = part.split(">", 1)[0].lstrip("<\n")
        lines = [ln.split("//")[0].strip() for ln in part.splitlines()[1:]]
        targets = set(re.findall(r"s_cbranch_execz (\w+)", part))

        def block(first, place):
            early = []
            for ln in lines[first:]:
                if LABEL.match(ln) or END.match(ln):
                    return
                if RESTORE.match(ln):
                    found.extend((name, place, e) for e in early)
                    return
                if ln.startswith(VECTOR) and not ln.startswith(HARMLESS):
                    early.append(ln)

        before = []                  # straight-line instructions since the last label, branch or mask change
        for i, ln in enumerate(lines):
            m = LABEL.match(ln)
            if m:
                if m.group(1) in targets:
                    block(i + 1, m.group(1))
                before = []
            elif ln.startswith("s_cbranch_execnz"):
                block(i + 1, "behind " + ln)
                before = []
            elif END.match(ln):
                before = []
            elif JOIN.match(ln):
                saves = []
                for e in reversed(before):
                    if SAVE.match(e):
                        saves.append(e)
                    elif SCALAR_COPY.match(e):
                        found.extend((name, "before " + ln, s) for s in saves)
                        saves = []
                    elif not WAIT.match(e):
                        break
                before = []
            elif " exec, " in ln or "saveexec" in ln:
                before = []
            else:
                before.append(ln)
    return found


def code_objects(path):
    """llvm-objdump's text of each gfx950 code object in a library."""
    with tempfile.TemporaryDirectory() as tmp:
        name = os.path.basename(path)
        os.symlink(os.path.abspath(path), os.path.join(tmp, name))
        subprocess.run([OBJDUMP, "--offloading", name], cwd=tmp, check=True, capture_output=True)
        for obj in sorted(p for p in os.listdir(tmp) if p.endswith("gfx950")):
            yield subprocess.run([OBJDUMP, "-d", "--symbolize-operands", "--no-show-raw-insn", "--no-leading-addr",
                                  obj], cwd=tmp, check=True, capture_output=True, text=True).stdout


def check(path):
    """(kernels looked at, faults found) of a library"""
    kernels, found = 0, []
    for asm in code_objects(path):
        kernels += asm.count("\n<_Z")
        found += early_vector_writes(asm)
    return kernels, found


def main(paths):
    status = 0
    for path in paths:
        kernels, found = check(path)
        if not kernels:
            print(f"check_isa: no gfx950 kernels in {path}", file=sys.stderr)
            status = 1
        for name, place, ins in found:
            print(f"check_isa: {path}: {name}: {place}: {ins}: ahead of the execution mask's restore",
                  file=sys.stderr)
            status = 1
    return status


if __name__ == "__main__":
    sys.exit(main(sys.argv[1:]))

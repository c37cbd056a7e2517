"""Wait states around the matrix instructions of the built library: the hardware does not
interlock a matrix instruction with the vector instructions beside it, and the compiler
inserts the wait states only around instructions it forms itself (not around inline
assembly).  The library's gfx950 code is listed and read in program order:

- a vector instruction's result is read by a matrix or DPP instruction after at least 2 wait
  states;
- the SrcC registers of v_mfma_f32_16x16x32_f16 (4 passes) are overwritten by a vector
  instruction after at least 3.

Every other instruction counts for one wait state, s_nop N for N + 1."""
import os
import re
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
LIB = os.path.join(os.path.dirname(HERE), "mc_kernel_amd", "libmck.so")
OBJDUMP = os.path.join(os.environ.get("ROCM_PATH", "/opt/rocm"), "llvm", "bin", "llvm-objdump")

REG = re.compile(r"^[-|]*v(?:\[(\d+):(\d+)\]|(\d+))")


def _regs(operand):
    m = REG.match(operand)
    if not m:
        return ()
    return range(int(m[1]), int(m[2]) + 1) if m[1] else (int(m[3]),)


def hazards(listing):
    """(function, kind, instruction, wait states) of every pair that is too close, and the
    number of matrix instructions"""
    found, nmfma, pos, written, recent, fn = [], 0, 0, {}, [], ""
    for line in listing:
        if line.startswith("<"):
            fn, written, recent = line[1:line.rindex(">")], {}, []
            continue
        op, _, rest = line.split("//")[0].strip().partition(" ")
        if not op.startswith(("v_", "s_nop")):
            pos += 1
            continue
        if op == "s_nop":
            pos += int(rest) + 1
            continue
        ops = [o.strip() for o in re.split(r",(?![^\[]*\])", rest)]
        mfma = op.startswith("v_mfma")
        dpp = "_dpp" in op or "row_" in rest or "quad_perm" in rest
        if mfma or dpp:
            w = [pos - written[q] - 1 for o in ops[1:4] for q in _regs(o) if q in written]
            if w and min(w) < 2:
                found.append((fn, "read", op, min(w)))
        if mfma:
            nmfma += 1
            if op == "v_mfma_f32_16x16x32_f16":
                recent = recent[-3:] + [(pos, set(_regs(ops[3])))]
        elif not op.startswith(("v_cmp", "v_readlane", "v_readfirstlane")):
            for q in _regs(ops[0]):
                written[q] = pos
                found += [(fn, "overwrite", op, pos - p - 1) for p, c in recent if q in c and pos - p - 1 < 3]
        pos += 1
    return found, nmfma


def test_reader_sees_each_kind():
    """the reader on listings with known distances"""
    f = "<kernel>:\n"
    m = "v_mfma_f32_16x16x32_f16 v[0:3], v[8:11], v[12:15], v[0:3]\n"
    far = f + "v_add_f32_e32 v9, v1, v2\ns_nop 1\n" + m
    near = f + "v_add_f32_e32 v9, v1, v2\ns_nop 0\n" + m
    assert hazards(far.splitlines()) == ([], 1)
    assert hazards(near.splitlines())[0] == [("kernel", "read", "v_mfma_f32_16x16x32_f16", 1)]
    over = f + m + "s_nop 1\nv_mov_b32_e32 v2, v20\n"
    assert hazards(over.splitlines())[0] == [("kernel", "overwrite", "v_mov_b32_e32", 2)]
    assert hazards((f + m + "s_nop 2\nv_mov_b32_e32 v2, v20\n").splitlines()) == ([], 1)
    dpp = f + "v_add_f32_e32 v9, v1, v2\nv_mov_b32_dpp v3, v9 row_ror:4 row_mask:0xf bank_mask:0xf\n"
    assert hazards(dpp.splitlines())[0] == [("kernel", "read", "v_mov_b32_dpp", 0)]


def test_wait_states(tmp_path):
    if not os.path.exists(OBJDUMP):
        pytest.skip("no llvm-objdump")
    if not os.path.exists(LIB):
        from mc_kernel_amd import build
        build.build_hip(force=False)
    shutil.copy(LIB, tmp_path / "libmck.so")
    subprocess.run([OBJDUMP, "--offloading", "libmck.so"], cwd=tmp_path, check=True, stdout=subprocess.DEVNULL)
    objs = [f for f in os.listdir(tmp_path) if "gfx950" in f]
    assert objs
    nmfma = 0
    for o in objs:
        out = subprocess.run([OBJDUMP, "-d", "--no-show-raw-insn", "--no-leading-addr", o], cwd=tmp_path, check=True,
                             stdout=subprocess.PIPE, text=True).stdout
        found, n = hazards(out.splitlines())
        nmfma += n
        assert not found, (len(found), found[:4])
    assert nmfma > 1000

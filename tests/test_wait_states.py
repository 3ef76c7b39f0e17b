"""Wait states of the built device code.

On gfx950 a VALU instruction that reads a mask or carry (an SGPR pair or vcc)
stands at least two wait states behind the VALU instruction that wrote it, and
a DPP instruction as far behind the VALU instruction that wrote its source
register: that is the distance hipcc keeps in its own code.  It does not look
into asm blocks, so the library's code objects are disassembled and every such
pair is measured along the straight line.
"""
import glob
import os
import re
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
LIB = os.path.join(ROOT, "velodb_amd", "libvelodb_amd.so")
OBJDUMP = "/opt/rocm/llvm/bin/llvm-objdump"

WAIT = 2
_SGPR = re.compile(r"\bs\[(\d+):(\d+)\]|\bs(\d+)\b|\b(vcc)\b")
_VGPR = re.compile(r"\bv\[(\d+):(\d+)\]|\bv(\d+)\b")
# carry instructions: vdst, then the carry written, then the operands read
_TWO_DST = re.compile(r"v_(?:add|sub|subrev|addc|subb|subbrev)_co_|v_div_scale|v_mad_[iu]64")


def _regs(pattern, text, kind):
    out = []
    for m in pattern.finditer(text):
        if m.group(1):
            out.extend(kind + str(i) for i in range(int(m.group(1)), int(m.group(2)) + 1))
        elif m.group(3):
            out.append(kind + m.group(3))
        else:
            out.append("vcc")
    return out


def short_waits(lines):
    """(function, instruction, wait states) of every read that comes too early."""
    found, name, clock, wrote = [], "", 0, {}
    for line in lines:
        if line.endswith(">:"):
            name, wrote = line.split("<")[-1][:-2], {}
            continue
        op, _, args = line.partition("//")[0].strip().partition(" ")
        if not op:
            continue
        if op == "s_nop":
            clock += int(args, 0) + 1
            continue
        clock += 1
        if op.startswith("s_"):
            for r in _regs(_SGPR, args.split(",")[0], "s"):
                wrote.pop(r, None)  # written by a scalar instruction: the hardware waits
            continue
        if not op.startswith("v_"):
            continue
        operands = args.split(",")
        n_dst = 2 if _TWO_DST.match(op) else 1
        dst, src = ",".join(operands[:n_dst]), ",".join(operands[n_dst:])
        read = _regs(_SGPR, src, "s")
        if op.endswith("_dpp"):
            read += _regs(_VGPR, operands[n_dst], "v")
        waits = min((clock - wrote[r] - 1 for r in read if r in wrote), default=WAIT)
        if waits < WAIT:
            found.append((name, line.strip(), waits))
        written = _regs(_SGPR, dst, "s") + _regs(_VGPR, operands[0], "v")
        if op.startswith("v_cmp") and op.endswith("_e32"):
            written.append("vcc")
        for r in written:
            wrote[r] = clock
    return found


@pytest.mark.parametrize("code,count", [
    ("v_sub_co_u32_e64 v0, s[2:3], v1, v2\nv_subb_co_u32_e64 v0, s[2:3], v3, v4, s[2:3]", 1),
    ("v_sub_co_u32_e64 v0, s[2:3], v1, v2\ns_nop 1\nv_subb_co_u32_e64 v0, s[2:3], v3, v4, s[2:3]", 0),
    ("v_sub_co_u32_e64 v0, s[2:3], v1, v2\nv_mov_b32_e32 v9, v8\ns_nop 0\n"
     "v_subb_co_u32_e64 v0, s[2:3], v3, v4, s[2:3]", 0),
    ("v_cmp_lt_u32_e64 s[4:5], v1, v2\nv_mov_b32_e32 v9, v8\nv_cndmask_b32_e64 v0, v1, v2, s[4:5]", 1),
    ("v_cmp_lt_u32_e32 vcc, v1, v2\nv_cndmask_b32_e32 v0, v1, v2, vcc", 1),
    ("v_cmp_lt_u32_e64 s[4:5], v1, v2\ns_mov_b64 s[4:5], s[4:5]\nv_cndmask_b32_e64 v0, v1, v2, s[4:5]", 0),
    ("v_readlane_b32 s4, v7, 3\nv_cndmask_b32_e64 v0, v1, v2, s[4:5]", 1),
    ("v_mov_b32_e32 v3, v8\nv_mov_b32_dpp v4, v3 quad_perm:[1,0,3,2] row_mask:0xf bank_mask:0xf", 1),
    ("v_mov_b32_e32 v3, v8\ns_nop 1\nv_mov_b32_dpp v4, v3 quad_perm:[1,0,3,2] row_mask:0xf bank_mask:0xf", 0),
    ("v_sub_co_u32_dpp v4, vcc, v1, v1 quad_perm:[1,0,3,2] row_mask:0xf bank_mask:0xf\n"
     "v_subb_co_u32_dpp v4, vcc, v2, v2, vcc quad_perm:[1,0,3,2] row_mask:0xf bank_mask:0xf", 1),
])
def test_short_waits_are_found(code, count):
    assert len(short_waits(code.split("\n"))) == count


def test_library_keeps_the_wait_states(tmp_path):
    if not os.path.exists(OBJDUMP) or not os.path.exists(LIB):
        pytest.skip("no disassembler or no built library")
    lib = shutil.copy(LIB, tmp_path)
    subprocess.check_call([OBJDUMP, "--offloading", os.path.basename(lib)], cwd=tmp_path, stdout=subprocess.DEVNULL)
    objects = glob.glob(os.path.join(tmp_path, "*gfx950*"))
    assert objects
    for obj in objects:
        with subprocess.Popen([OBJDUMP, "-d", "--no-show-raw-insn", obj], stdout=subprocess.PIPE, text=True) as p:
            found = short_waits(map(str.rstrip, p.stdout))
        assert p.returncode == 0
        assert not found, f"{len(found)} reads too early, the first: {found[:3]}"

"""The built kernels keep the hardware's distance between a vector instruction
that writes a scalar register (a compare's lane mask, say) and a vector
instruction that reads it: two wait states, without which the reader may see
the register's former bits.  The compiler fills them in its own code but not
between inline asm statements, so this reads the machine code of every kernel
in the library in program order and counts them."""
import os
import re
import shutil
import struct
import subprocess

import pytest

from conftest import ROOT

LIB = os.path.join(ROOT, "swm_amd", "libswmgpu.so")
OBJDUMP = shutil.which("llvm-objdump") or "/opt/rocm/llvm/bin/llvm-objdump"
WAIT_STATES = 2
SGPR = re.compile(r"-?\|?(?:(vcc)(?:_lo|_hi)?|s(\d+)|s\[(\d+):(\d+)\])\|?$")
# sdst is the second operand: carries, div_scale and the wide multiply-adds
TWO_DST = re.compile(r"v_(add|sub|subrev|addc|subb|subbrev)_co_|v_div_scale_|v_mad_[iu]64_[iu]32")


def gfx950_code(lib):
    """The gfx950 code object of the library's offload bundle."""
    data = open(lib, "rb").read()
    at = data.index(b"__CLANG_OFFLOAD_BUNDLE__")
    p = at + 24
    n, = struct.unpack_from("<Q", data, p)
    p += 8
    for _ in range(n):
        off, size, name_len = struct.unpack_from("<QQQ", data, p)
        name = data[p + 24:p + 24 + name_len].decode()
        p += 24 + name_len
        if name.endswith("gfx950"):
            return data[at + off:at + off + size]
    raise AssertionError("no gfx950 code in the library")


def sgprs(operand):
    m = SGPR.match(operand.strip())
    if not m:
        return ()
    if m[1]:
        return ("vcc",)
    return range(int(m[2]), int(m[2]) + 1) if m[2] else range(int(m[3]), int(m[4]) + 1)


def close_reads(lines):
    """(kernel, write, read, wait states) of every pair that is too close."""
    found, kernel, written, now = [], None, {}, 0
    for line in lines:
        if not line.startswith("\t"):
            if line.endswith(">:\n"):
                kernel, written = line.split("<")[1][:-3], {}
            continue
        ins = line.split("//")[0].strip()
        if ins.startswith("s_nop"):
            now += int(ins.split()[1], 0) + 1
            continue
        now += 1
        if "vcc" not in ins and " s" not in ins:
            continue
        op, _, rest = ins.partition(" ")
        ops = rest.split(",")
        if op.startswith("s_"):      # a scalar instruction's own write is another matter
            for r in sgprs(ops[0]):
                written.pop(r, None)
        elif op.startswith("v_"):
            dst = ops[1:2] if TWO_DST.match(op) else ops[:1] if op.startswith(("v_cmp", "v_read")) else []
            for x in ops[2 if TWO_DST.match(op) else 1:]:
                for r in sgprs(x):
                    if r in written and now - written[r][0] - 1 < WAIT_STATES:
                        found.append((kernel, written[r][1], ins, now - written[r][0] - 1))
            for x in dst:
                for r in sgprs(x):
                    written[r] = (now, ins)
    return found


def test_the_count_finds_a_close_pair():
    pair = ["0 <k>:\n", "\tv_cmp_class_f64_e64 s[4:5], v[2:3], s9 // 0\n", "\ts_nop 0\n",
            "\tv_cndmask_b32_e64 v0, v1, v2, s[4:5]\n"]
    assert [f[3] for f in close_reads(pair)] == [1, 1]   # one for each register of the mask
    assert not close_reads(pair[:2] + ["\ts_nop 1\n"] + pair[3:])
    assert not close_reads(pair[:2] + ["\ts_mov_b64 s[4:5], exec\n"] + pair[3:])


def test_masks_are_read_two_wait_states_after_their_write(tmp_path):
    if not os.path.exists(LIB) or not os.path.exists(OBJDUMP):
        pytest.skip("no library or no disassembler")
    code = tmp_path / "gfx950.co"
    code.write_bytes(gfx950_code(LIB))
    with subprocess.Popen([OBJDUMP, "-d", "--no-show-raw-insn", str(code)], stdout=subprocess.PIPE, text=True) as p:
        found = close_reads(p.stdout)
    assert p.returncode == 0
    assert not found, (len(found), found[:3])

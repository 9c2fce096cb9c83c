"""The built library's gfx950 code: the wait states that direct global-to-LDS
loads need.  The kernels issue these loads from inline assembly, where the
compiler inserts no waits of its own: one state between a scalar write of M0
(the LDS address) and the load, five between a vector instruction's write of
the load's scalar base and the load."""
import os
import re
import struct
import subprocess
import tempfile

import pytest

from wnw_amd import _lib

LLVM = "/opt/rocm/llvm/bin"


def _registers(operands):
    regs = set()
    for a, b in re.findall(r"\bs\[(\d+):(\d+)\]", operands):
        regs |= set(range(int(a), int(b) + 1))
    return regs | {int(x) for x in re.findall(r"\bs(\d+)\b", operands)}


def _code_objects(path, tmp):
    fat = os.path.join(tmp, "fat.bin")
    subprocess.run([f"{LLVM}/llvm-objcopy", f"--dump-section=.hip_fatbin={fat}", path, os.path.join(tmp, "rest")],
                   check=True)
    data = open(fat, "rb").read()
    for m in re.finditer(b"__CLANG_OFFLOAD_BUNDLE__", data):
        at = m.start() + 32
        for _ in range(struct.unpack_from("<Q", data, m.start() + 24)[0]):
            off, size, n = struct.unpack_from("<QQQ", data, at)
            if b"gfx950" in data[at + 24:at + 24 + n] and size:
                yield data[m.start() + off:m.start() + off + size]
            at += 24 + n


def lds_load_hazards(lines):
    """(loads, [(kernel, instruction, load)]) of a disassembly: the loads
    whose M0 or scalar base was written too few wait states before."""
    loads, bad, kernel, before = 0, [], "", []
    for line in lines:
        op = line.split("//")[0].strip()
        if op.endswith(">:"):
            kernel, before = op, []
        elif op:
            if op.startswith("global_load_lds"):
                loads += 1
                base, states = _registers(op.split(None, 1)[1]), 0
                for prev in reversed(before):
                    name, _, args = prev.partition(" ")
                    written = ",".join(args.split(",")[:2 if "_co_" in name else 1])
                    if states < 1 and name.startswith("s_") and re.match(r"\s*m0\b", args):
                        bad.append((kernel, prev, op))
                    if states < 5 and name.startswith("v_") and _registers(written) & base:
                        bad.append((kernel, prev, op))
                    states += int(args) + 1 if name == "s_nop" else 1
                    if states >= 5:
                        break
            before = before[-8:] + [op]
    return loads, bad


def test_the_check_itself():
    ok = ["v_readfirstlane_b32 s1, v3", "s_mov_b32 s4, m0", "s_mov_b32 m0, s2", "s_nop 2",
          "global_load_lds_dwordx4 v2, s[0:1] nt"]
    assert lds_load_hazards(ok) == (1, [])
    assert len(lds_load_hazards(ok[:3] + ["s_nop 0"] + ok[4:])[1]) == 1  # the base, three states before
    assert len(lds_load_hazards(ok[1:3] + ok[4:])[1]) == 1  # M0, none
    assert len(lds_load_hazards(["v_add_co_u32_e64 v1, s[0:1], v2, v3"] + ok[4:])[1]) == 1


@pytest.mark.skipif(not os.path.exists(f"{LLVM}/llvm-objdump"), reason="no llvm-objdump")
def test_lds_loads_wait_for_their_scalars():
    loads, bad = 0, []
    with tempfile.TemporaryDirectory() as tmp:
        for i, code in enumerate(_code_objects(_lib.LIB_PATH, tmp)):
            path = os.path.join(tmp, f"{i}.elf")
            with open(path, "wb") as f:
                f.write(code)
            text = subprocess.run([f"{LLVM}/llvm-objdump", "-d", "--no-show-raw-insn", "--no-leading-addr", path],
                                  check=True, capture_output=True, text=True).stdout
            n, b = lds_load_hazards(text.splitlines())
            loads += n
            bad += b
    assert loads > 0
    assert not bad, (len(bad), bad[:3])

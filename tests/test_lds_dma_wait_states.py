"""Wait states before the loads to LDS, read from the machine code of the built library.

Two dependencies that gfx9-family hardware does not interlock: a scalar write of M0 and a load to
LDS, which takes its LDS address from M0 (one wait state), and a vector instruction's write of
a scalar register and a memory instruction that reads it as its base (five). The compiler
inserts them between instructions of its own; these loads stand in inline asm, where it does not.
"""
import re
import struct
import subprocess
from pathlib import Path

import pytest

from geoweave_amd import build as gw_build

OBJDUMP = Path("/opt/rocm/llvm/bin/llvm-objdump")
MAGIC = b"__CLANG_OFFLOAD_BUNDLE__"


def _device_code(lib: bytes):
    """The gfx950 code objects of the offload bundles in a shared library."""
    at = lib.find(MAGIC)
    while at >= 0:
        (n,) = struct.unpack_from("<Q", lib, at + len(MAGIC))
        p = at + len(MAGIC) + 8
        for _ in range(n if n < 16 else 0):
            off, size, idlen = struct.unpack_from("<QQQ", lib, p)
            name = lib[p + 24:p + 24 + idlen]
            p += 24 + idlen
            if name.endswith(b"gfx950") and size:
                yield lib[at + off:at + off + size]
        at = lib.find(MAGIC, at + 1)


def _sregs(operand: str):
    m = re.fullmatch(r"s\[(\d+):(\d+)\]", operand)
    if m:
        return set(range(int(m[1]), int(m[2]) + 1))
    m = re.fullmatch(r"s(\d+)", operand)
    return {int(m[1])} if m else set()


def _is_lds_load(ops):
    return "_load_lds_" in ops[0] or (ops[0].startswith("buffer_load") and "lds" in ops)


def _hazards(lines):
    """(number of loads to LDS, those with too few wait states) of disassembled lines."""
    loads, found, last = 0, [], []
    for line in lines:
        text = line.split("//")[0].strip()
        if not text or text.endswith(":"):
            if text:
                last = []
            continue
        ops = re.split(r"[ ,]+", text)
        if _is_lds_load(ops):
            loads += 1
            base = set().union(*(_sregs(x) for x in ops[1:]))
            states, m0 = 0, False
            for prev in reversed(last):
                if not m0 and prev[0].startswith("s_") and prev[1:2] == ["m0"]:
                    m0 = True
                    if states < 1:
                        found.append((prev, ops))
                if prev[0].startswith("v_") and len(prev) > 1 and _sregs(prev[1]) & base and states < 5:
                    found.append((prev, ops))
                states += int(prev[1], 0) + 1 if prev[0] == "s_nop" else 1
        last = last[-7:] + [ops]
    return loads, found


def test_the_check_sees_both_hazards():
    move, base, load = "s_mov_b32 m0, s4", "v_readfirstlane_b32 s8, v1", "global_load_lds_dwordx4 v2, s[8:9]"
    assert _hazards([move, load])[1] and not _hazards([move, "s_nop 0", load])[1]
    assert _hazards([base, "s_nop 3", load])[1] and not _hazards([base, "s_nop 4", load])[1]
    assert _hazards(["s_nop 0", base, move, "s_nop 2", load])[1]


def test_no_load_to_lds_lacks_its_wait_states(tmp_path):
    if not OBJDUMP.exists():
        pytest.skip("no llvm-objdump")
    lib = gw_build.LIB_PATH if gw_build.LIB_PATH.exists() else gw_build.build()
    loads, found = 0, []
    for i, code in enumerate(_device_code(lib.read_bytes())):
        path = tmp_path / f"{i}.co"
        path.write_bytes(code)
        with subprocess.Popen([str(OBJDUMP), "-d", "--no-show-raw-insn", str(path)], stdout=subprocess.PIPE, text=True) as p:
            n, bad = _hazards(p.stdout)
        assert p.returncode == 0
        loads, found = loads + n, found + bad
    assert loads > 100
    assert not found, f"{len(found)} of {loads} loads, first: {found[0]}"

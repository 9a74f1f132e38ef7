"""The wait state between a scalar write of M0 and a load from global memory straight into LDS.

The loads of ``pycc_amd/csrc/gemm_plain.hip`` and ``split16.hip`` take their LDS address from M0, which the
hardware needs one wait state to see after a scalar instruction wrote it; in inline assembly the compiler does
not add it. Checked in the gfx950 code of the built library, whoever wrote the instructions."""
import os
import re
import shutil
import struct
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
LIB = os.path.join(ROOT, "pycc_amd", "libccx.so")
OBJDUMP = "/opt/rocm/llvm/bin/llvm-objdump"
MAGIC = b"__CLANG_OFFLOAD_BUNDLE__"
pytestmark = pytest.mark.skipif(not os.path.exists(LIB) or shutil.which(OBJDUMP) is None,
                                reason="library not built, or no disassembler")


def _code_objects():
    """The GPU code objects of the library: a bundle per source file, each a table of (offset, size, name)."""
    data = open(LIB, "rb").read()
    at = data.find(MAGIC)
    while at >= 0:
        n, = struct.unpack_from("<Q", data, at + len(MAGIC))
        p = at + len(MAGIC) + 8
        for _ in range(n):
            off, size, length = struct.unpack_from("<QQQ", data, p)
            name = data[p + 24:p + 24 + length].decode()
            p += 24 + length
            if "gfx950" in name and size:
                yield data[at + off:at + off + size]
        at = data.find(MAGIC, p)


def unprotected(lines):
    """Pairs (write of M0, load into LDS) with no instruction in between."""
    bad, last = [], ""
    for line in lines:
        ins = line.split("//")[0].strip()
        if not ins or ins.endswith(":"):
            continue
        if re.match(r"(global_load_lds|buffer_load\S*.* lds)", ins) and re.match(r"s_\S+ m0,", last):
            bad.append((last, ins))
        last = ins
    return bad


def test_the_check_sees_a_missing_wait_state():
    load = "global_load_lds_dwordx4 v[0:1], off"
    assert unprotected(["s_mov_b32 m0, s4 // 0", load]) == [("s_mov_b32 m0, s4", load)]
    assert unprotected(["s_mov_b32 m0, s4", "s_nop 0", load, load]) == []


def test_every_load_into_lds_waits_for_m0(tmp_path):
    loads = 0
    for i, obj in enumerate(_code_objects()):
        path = tmp_path / ("code%d.o" % i)
        path.write_bytes(obj)
        text = subprocess.run([OBJDUMP, "-d", "--no-show-raw-insn", "--mcpu=gfx950", str(path)], capture_output=True, text=True,
                              check=True).stdout.splitlines()
        loads += sum("global_load_lds" in t for t in text)
        bad = unprotected(text)
        assert not bad, (len(bad), bad[0])
    assert loads > 0

"""Loads from memory to LDS take their destination from M0 and need a wait state behind a scalar write of it (and, as every
memory instruction, five behind a vector instruction's write of a scalar that they read).  They are written in assembly, which the
compiler's own insertion of wait states does not look into: checked in the code of the built library."""
import os
import re
import struct
import subprocess

import pytest

from kitty_amd import _lib

OBJDUMP = "/opt/rocm/llvm/bin/llvm-objdump"
MAGIC = b"__CLANG_OFFLOAD_BUNDLE__"


def _device_objects(data):
    """The gfx950 code objects of a library's offload bundles."""
    at = data.find(MAGIC)
    while at >= 0:
        p = at + len(MAGIC)
        (n,) = struct.unpack_from("<Q", data, p)
        p += 8
        for _ in range(n):
            offset, size, id_len = struct.unpack_from("<QQQ", data, p)
            name = data[p + 24:p + 24 + id_len]
            p += 24 + id_len
            if b"gfx950" in name and size:
                yield data[at + offset:at + offset + size]
        at = data.find(MAGIC, at + len(MAGIC))


def _scalars(text):
    """The scalar registers a piece of operand text names."""
    out = {"m0"} if re.search(r"\bm0\b", text) else set()
    for a, b in re.findall(r"\bs(?:\[(\d+):|(\d+)\b)", text):
        out.add(int(a or b))
    for a, b in re.findall(r"\bs\[(\d+):(\d+)\]", text):
        out.update(range(int(a), int(b) + 1))
    return out


def hazards(lines):
    """(loads to LDS, those less than a wait state behind a scalar write of M0 or five behind a vector instruction's write of a scalar
    that they read)"""
    loads, bad, before = 0, [], []          # before: (what it is, the scalars it writes), a wait state each, the last one first
    for line in lines:
        m = re.match(r"\s+([a-z]\w+)\s*(.*?)\s*(//.*)?$", line)
        if not m:
            continue
        op, args = m.group(1), m.group(2)
        if "load_lds" in op or (op.startswith("buffer_load") and re.search(r"\blds\b", args)):
            loads += 1
            reads = _scalars(args) | {"m0"}
            for i, (what, writes) in enumerate(before):
                if (i < 1 and what[0] == "s" and "m0" in writes) or (what[0] == "v" and writes & reads):
                    bad.append(what + " / " + line.strip())
        states = int(args, 0) + 1 if op == "s_nop" else 1
        writes = set() if op == "s_nop" or op[0] not in "sv" else _scalars(args.split(",")[0])
        before = ([(op + " " + args, writes)] + [("s_nop", set())] * (states - 1) + before)[:5]
    return loads, bad


def test_reader():
    def load(*before):
        return hazards(["\t" + x + "   // 000: AB" for x in before + ("global_load_lds_dword v1, s[2:3] nt",)])

    assert load("s_mov_b32 m0, s4")[0] == 1 and len(load("s_mov_b32 m0, s4")[1]) == 1
    assert load("s_mov_b32 m0, s4", "s_nop 0") == (1, []) and load("s_mov_b32 m0, s4", "v_mov_b32_e32 v1, v2") == (1, [])
    assert len(load("v_readfirstlane_b32 s3, v9", "s_mov_b32 m0, s4", "s_nop 2")[1]) == 1
    assert load("v_readfirstlane_b32 s3, v9", "s_mov_b32 m0, s4", "s_nop 3") == (1, [])
    assert load("v_readfirstlane_b32 s5, v9", "s_nop 0") == (1, [])


@pytest.mark.skipif(not os.path.exists(OBJDUMP) or not os.path.exists(_lib.LIB_PATH), reason="needs the built library and llvm-objdump")
def test_wait_states(tmp_path):
    with open(_lib.LIB_PATH, "rb") as f:
        data = f.read()
    loads = 0
    for i, obj in enumerate(_device_objects(data)):
        path = tmp_path / f"{i}.o"
        path.write_bytes(obj)
        text = subprocess.run([OBJDUMP, "-d", "--mcpu=gfx950", str(path)], check=True, capture_output=True, text=True).stdout
        n, bad = hazards(text.splitlines())
        loads += n
        assert not bad, f"{len(bad)} of {n} loads, for instance {bad[0]}"
    assert loads > 100

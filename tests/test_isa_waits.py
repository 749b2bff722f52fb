"""The built device code keeps the wait states that the hardware asks for and the
compiler does not see across inline assembly: a buffer instruction reads a scalar
register no sooner than 5 wait states after a vector instruction wrote it."""
import os
import re
import struct
import subprocess

import pytest

from nsw import _lib

OBJDUMP = "/opt/rocm/llvm/bin/llvm-objdump"
MAGIC = b"__CLANG_OFFLOAD_BUNDLE__"
WAIT = 5


def _device_objects(path):
    data = open(path, "rb").read()
    at = data.find(MAGIC)
    while at >= 0:
        n, = struct.unpack_from("<Q", data, at + len(MAGIC))
        p = at + len(MAGIC) + 8
        for _ in range(n):
            off, size, idlen = struct.unpack_from("<QQQ", data, p)
            ident = data[p + 24:p + 24 + idlen]
            p += 24 + idlen
            if b"gfx950" in ident and size:
                yield data[at + off:at + off + size]
        at = data.find(MAGIC, at + 1)


def _sgprs(text):
    regs = set()
    for a, b in re.findall(r"\bs\[(\d+):(\d+)\]", text):
        regs.update(range(int(a), int(b) + 1))
    regs.update(int(a) for a in re.findall(r"\bs(\d+)\b", text))
    return regs


def too_close(lines):
    """(writer, reader) pairs of a listing with fewer than WAIT wait states between."""
    recent, pairs = [], []              # (instruction, scalar registers it wrote with the vector unit), per wait state
    for line in lines:
        ins = line.split("//")[0].strip()
        op = ins.split(" ", 1)[0]
        if op.startswith("buffer_"):
            used = _sgprs(ins)
            pairs += [(w, ins) for w, regs in recent if regs & used]
        wrote = set()
        if op.startswith(("v_readfirstlane", "v_readlane", "v_cmp")):
            wrote = _sgprs(ins.split(" ", 1)[1].split(",")[0])
        states = int(ins.split()[1], 0) + 1 if op == "s_nop" else 1
        recent = (recent + [(ins, wrote)] + [("", set())] * (states - 1))[-WAIT:]
    return pairs


def test_the_scan_sees_a_pair():
    read = "buffer_load_dwordx4 v82, s[20:23], s12 offen lds"
    near = ["v_readfirstlane_b32 s22, v138 // 0000: 1", "s_mov_b32 m0, s13", "s_nop 0", read]
    assert len(too_close(near)) == 1
    assert not too_close(near[:2] + ["s_nop 3", read])
    assert not too_close(["v_readfirstlane_b32 s24, v138", read])


@pytest.mark.skipif(not os.path.exists(OBJDUMP), reason="no disassembler for the device code")
def test_buffer_instructions_wait_for_their_scalars(tmp_path):
    found = buffers = 0
    for i, obj in enumerate(_device_objects(_lib.LIB_PATH)):
        f = tmp_path / f"{i}.o"
        f.write_bytes(obj)
        r = subprocess.run([OBJDUMP, "-d", "--no-show-raw-insn", "--mcpu=gfx950", str(f)], capture_output=True, text=True, check=True)
        lines = [l for l in r.stdout.splitlines() if l.startswith("\t")]
        buffers += sum("buffer_load" in l for l in lines)
        pairs = too_close(lines)
        found += len(pairs)
        for w, b in pairs[:3]:
            print(f"object {i}: {w} / {b}")
    assert buffers > 1000, "no device code found"
    assert found == 0

"""Registers and scratch of the built kernels, from the metadata note of the
library's gfx950 code objects (no GPU): only the interpreter, whose codecs are
called out of line, uses scratch memory."""
import struct

import msgpack

from zosimos_amd import build

INTERPRETER = ("k_pointwise", "k_resample", "k_batch")


def _note(elf):
    """The AMDGPU metadata (note type 32) of a code object."""
    assert elf[:4] == b"\x7fELF"
    phoff, = struct.unpack_from("<Q", elf, 32)
    size, count = struct.unpack_from("<HH", elf, 54)
    for i in range(count):
        kind, _, off, _, _, n = struct.unpack_from("<IIQQQQ", elf, phoff + i * size)
        at, end = off, off + n
        while kind == 4 and at < end:
            name, desc, note = struct.unpack_from("<III", elf, at)
            at += 12 + (name + 3) // 4 * 4
            if note == 32:
                return msgpack.unpackb(elf[at:at + desc])
            at += (desc + 3) // 4 * 4
    raise AssertionError("no metadata note")


def _kernels():
    with open(build.LIB, "rb") as f:
        lib = f.read()
    magic, out = b"__CLANG_OFFLOAD_BUNDLE__", []
    start = lib.find(magic)
    while start >= 0:
        entries, = struct.unpack_from("<Q", lib, start + 24)
        at = start + 32
        for _ in range(entries):
            off, n, text = struct.unpack_from("<QQQ", lib, at)
            if n and b"gfx950" in lib[at + 24:at + 24 + text]:
                out += _note(lib[start + off:start + off + n])["amdhsa.kernels"]
            at += 24 + text
        start = lib.find(magic, start + 1)
    return out


def test_only_the_interpreter_uses_scratch():
    kernels = _kernels()
    assert any("k_any" in k[".name"] for k in kernels) and any("k_warp" in k[".name"] for k in kernels)
    held = {k[".name"]: k[".private_segment_fixed_size"] for k in kernels
            if k[".private_segment_fixed_size"] and not any(i in k[".name"] for i in INTERPRETER)}
    assert not held

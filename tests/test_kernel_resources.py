"""Scratch memory and spilled registers of step kernels whose register budget is tight, from the
metadata notes of the code objects in the built library (CPU only).  The bounds are what these
kernels need; a change that spills more slows them down without failing any other test."""
import struct

import msgpack
import pytest

from ecogen_amd import LIB_PATH


def _code_objects(blob):
    """ELF images of the clang offload bundles in the library."""
    magic = b"__CLANG_OFFLOAD_BUNDLE__"
    at = blob.find(magic)
    while at >= 0:
        n, = struct.unpack_from("<Q", blob, at + 24)
        pos = at + 32
        for _ in range(n):
            off, size, tlen = struct.unpack_from("<QQQ", blob, pos)
            target = blob[pos + 24:pos + 24 + tlen]
            pos += 24 + tlen
            if b"gfx950" in target:
                yield blob[at + off:at + off + size]
        at = blob.find(magic, at + 1)


def _metadata(elf):
    """The AMDGPU metadata note (type 32) of a code object."""
    phoff, = struct.unpack_from("<Q", elf, 32)
    phentsize, phnum = struct.unpack_from("<HH", elf, 54)
    for i in range(phnum):
        ptype, _, off, _, _, size = struct.unpack_from("<IIQQQQ", elf, phoff + i * phentsize)
        if ptype != 4:   # PT_NOTE
            continue
        pos, end = off, off + size
        while pos < end:
            nlen, dlen, kind = struct.unpack_from("<III", elf, pos)
            data = pos + 12 + (nlen + 3) // 4 * 4
            if kind == 32:
                return msgpack.unpackb(elf[data:data + dlen])
            pos = data + (dlen + 3) // 4 * 4
    raise AssertionError("code object without metadata")


@pytest.fixture(scope="module")
def kernels():
    found = {}
    with open(LIB_PATH, "rb") as f:
        for elf in _code_objects(f.read()):
            for k in _metadata(elf)["amdhsa.kernels"]:
                found[k[".name"]] = k
    assert found
    return found


def _step(model, nph, dim, second, real, learned, limiter, capture=False, tile=None):
    """Mangled template arguments of k_step (limiter -1: chosen at run time, -2: full-featured)."""
    lk = f"n{-limiter}" if limiter < 0 else str(limiter)
    tile = tile or {"d": 8, "f": 4}[real]
    return (f"6k_stepILi{model}ELi{nph}ELi{dim}ELb{int(second)}E{real}Lb{int(learned)}ELi{lk}ELb{int(capture)}"
            f"ELi{tile}EE")


PUEQ, UEQ, MINMOD = 1, 2, 1
# Second-order three-phase FP32 kernels with the limiter fixed hold each limited slope only
# where it is used: no scratch.  Finite-rate two-phase 3D FP64: f' in a copy of its own, 41 spills.
BOUNDS = [(_step(m, 3, 3, True, "f", learned, MINMOD), 0) for m in (PUEQ, UEQ) for learned in (False, True)] + \
         [(_step(UEQ, 2, 3, False, "d", False, -2), 48)]


@pytest.mark.parametrize("name,spills", BOUNDS)
def test_spilled_registers(kernels, name, spills):
    match = [k for n, k in kernels.items() if name in n]
    assert len(match) == 1, (name, len(match))
    assert match[0][".vgpr_spill_count"] <= spills
    if spills == 0:
        assert match[0][".private_segment_fixed_size"] == 0

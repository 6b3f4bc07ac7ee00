"""CPU: register spills of kernels whose speed rests on holding whole lines in
registers, read from the kernel metadata of the built library (the note that
the compiler writes beside each kernel)."""
from __future__ import annotations

import struct
from pathlib import Path

import pytest

msgpack = pytest.importorskip("msgpack")

LIB = Path(__file__).resolve().parents[1] / "genesis4_cuda_port_amd" / "_lib" / "libg4hip.so"
BUNDLE = b"__CLANG_OFFLOAD_BUNDLE__"


def _notes(elf: bytes):
    """amdhsa.kernels of one code object (ELF64 note type 32, MessagePack)."""
    shoff, = struct.unpack_from("<Q", elf, 0x28)
    entry, count = struct.unpack_from("<HH", elf, 0x3A)
    for i in range(count):
        sh = shoff + i * entry
        if struct.unpack_from("<I", elf, sh + 4)[0] != 7:  # SHT_NOTE
            continue
        at, size = struct.unpack_from("<QQ", elf, sh + 24)
        end = at + size
        while at < end:
            nname, ndesc, kind = struct.unpack_from("<III", elf, at)
            at += 12 + (nname + 3) // 4 * 4
            if kind == 32:
                yield from msgpack.unpackb(elf[at:at + ndesc])["amdhsa.kernels"]
            at += (ndesc + 3) // 4 * 4


def _kernels():
    data = LIB.read_bytes()
    at = data.find(BUNDLE)
    while at >= 0:
        count, = struct.unpack_from("<Q", data, at + 24)
        p = at + 32
        for _ in range(count):
            off, size, ntriple = struct.unpack_from("<QQQ", data, p)
            triple = data[p + 24:p + 24 + ntriple]
            p += 24 + ntriple
            if size and b"gfx950" in triple:
                yield from _notes(data[at + off:at + off + size])
        at = data.find(BUNDLE, at + 24)


@pytest.mark.parametrize("name,instances", [("fft_rows_half_kernel", 12),
                                            ("fft_cols_half_kernel", 12)])
def test_line_pairs_do_not_spill(name, instances):
    """Both passes of every transform-pair size, FP64 and MIXED: two lines per
    lane, no vector or scalar register in memory."""
    found = [k for k in _kernels() if name in k[".name"]]
    assert len(found) == instances
    for k in found:
        assert k[".vgpr_spill_count"] == 0 and k[".sgpr_spill_count"] == 0, k[".name"]

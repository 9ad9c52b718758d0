"""Registers of the built kernels, read from the code object metadata inside libboa_hip.so (no GPU)."""
import os
import struct

import pytest

from boa_amd import build


def _sections(elf: bytes):
    """name -> (type, contents) of a 64-bit little-endian ELF image's sections."""
    shoff, = struct.unpack_from("<Q", elf, 0x28)
    shentsize, shnum, shstrndx = struct.unpack_from("<HHH", elf, 0x3A)
    heads = [struct.unpack_from("<IIQQQQIIQQ", elf, shoff + i * shentsize) for i in range(shnum)]
    names = elf[heads[shstrndx][4]:heads[shstrndx][4] + heads[shstrndx][5]]
    return [(names[h[0]:names.index(b"\0", h[0])].decode(), h[1], elf[h[4]:h[4] + h[5]]) for h in heads]


def _code_objects(lib: bytes):
    """The gfx950 code objects of the library's offload bundles (one bundle per source file)."""
    magic = b"__CLANG_OFFLOAD_BUNDLE__"
    fat = next(c for n, _, c in _sections(lib) if n == ".hip_fatbin")
    at = fat.find(magic)
    while at >= 0:
        n, = struct.unpack_from("<Q", fat, at + 24)
        p = at + 32
        for _ in range(n):
            off, size, idlen = struct.unpack_from("<QQQ", fat, p)
            ident = fat[p + 24:p + 24 + idlen].decode()
            p += 24 + idlen
            if "gfx950" in ident:
                yield fat[at + off:at + off + size]
        at = fat.find(magic, at + 1)


def _unpack(b: bytes, i: int):
    """The MessagePack value at b[i], and where it ends (the types that code object metadata uses)."""
    t = b[i]
    i += 1
    if t < 0x80:
        return t, i
    if t in (0xC0, 0xC2, 0xC3):
        return {0xC0: None, 0xC2: False, 0xC3: True}[t], i
    if 0xCC <= t <= 0xD3:  # unsigned, then signed, of 1, 2, 4, 8 bytes
        n = 1 << ((t - 0xCC) & 3)
        return int.from_bytes(b[i:i + n], "big", signed=t >= 0xD0), i + n
    if 0xD9 <= t <= 0xDF:  # string, array, map with the length in 1 (string only), 2, 4 bytes
        n = {0xD9: 1, 0xDA: 2, 0xDB: 4, 0xDC: 2, 0xDD: 4, 0xDE: 2, 0xDF: 4}[t]
        kind, n, i = ("str" if t < 0xDC else "array" if t < 0xDE else "map"), int.from_bytes(b[i:i + n], "big"), i + n
    else:
        assert t < 0xC0, hex(t)
        kind, n = ("map", t & 15) if t < 0x90 else ("array", t & 15) if t < 0xA0 else ("str", t & 31)
    if kind == "str":
        return b[i:i + n].decode(), i + n
    out = []
    for _ in range(n * (2 if kind == "map" else 1)):
        v, i = _unpack(b, i)
        out.append(v)
    return (dict(zip(out[::2], out[1::2])) if kind == "map" else out), i


def _kernels():
    """Mangled kernel name -> its metadata."""
    lib = open(build.OUT, "rb").read()
    out = {}
    for co in _code_objects(lib):
        for _, kind, c in _sections(co):
            if kind != 7:  # SHT_NOTE
                continue
            namesz, descsz, ntype = struct.unpack_from("<III", c, 0)
            if ntype != 32:  # NT_AMDGPU_METADATA
                continue
            desc = c[12 + (namesz + 3) // 4 * 4:][:descsz]
            for k in _unpack(desc, 0)[0]["amdhsa.kernels"]:
                out[k[".name"]] = k
    return out


# Kernels of the compress and forward paths whose inner loops have no registers to spare: their launch bounds put them
# at or near the limit, and a spill is a round trip to scratch per K step.
@pytest.mark.parametrize("name", ["5k_ffnI", "8k_ffn512I", "7k_ffn16I", "7k_mixinI", "10k_mixin512I", "9k_head_xqI",
                                  "8k_head16I", "6k_scanI", "10k_scan_genI", "11k_scan_quadI"])
def test_compress_kernels_do_not_spill(name):
    """No form of the kernel keeps vector registers in scratch memory."""
    assert os.path.exists(build.OUT), "build first"
    found = {k: v for k, v in _kernels().items() if name in k}
    assert found, name
    bad = {k: (v[".vgpr_spill_count"], v[".private_segment_fixed_size"]) for k, v in found.items()
           if v[".vgpr_spill_count"] or v[".private_segment_fixed_size"]}
    assert not bad, bad

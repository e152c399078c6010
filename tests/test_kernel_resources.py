"""What the compiled gfx950 kernels ask of the machine, read from their descriptors in the built library (no GPU needed).

No kernel of the render loop may use scratch memory (a private segment): a k_shade variant that spilled registers to it
ended in a GPU memory fault when a captured graph launched it first, and that variant, the batched kernel without media, is
not compiled at all.
"""
import os
import re
import struct

import pytest

from vviewer_amd import build

MARK = b"__CLANG_OFFLOAD_BUNDLE__"


def _code_objects(data):
    """The gfx950 ELF images of the library's fat binaries (uncompressed clang offload bundles)."""
    at = data.find(MARK)
    while at >= 0:
        n, = struct.unpack_from("<Q", data, at + len(MARK))
        o = at + len(MARK) + 8
        for _ in range(n):
            off, size, ln = struct.unpack_from("<QQQ", data, o)
            name = data[o + 24:o + 24 + ln]
            o += 24 + ln
            if b"gfx950" in name and size:
                yield data[at + off:at + off + size]
        at = data.find(MARK, at + 1)


def _descriptors(elf):
    """{kernel: (LDS bytes, scratch bytes per lane)} from the 64-byte kernel descriptors, symbols `<kernel>.kd`."""
    shoff, = struct.unpack_from("<Q", elf, 40)
    shentsize, shnum = struct.unpack_from("<HH", elf, 58)
    sec = [struct.unpack_from("<IIQQQQIIQQ", elf, shoff + k * shentsize) for k in range(shnum)]
    out = {}
    for s in sec:
        if s[1] != 11:  # SHT_DYNSYM
            continue
        strtab = sec[s[6]]
        for k in range(s[5] // s[9]):
            name, _, _, shndx, value, size = struct.unpack_from("<IBBHQQ", elf, s[4] + k * s[9])
            a = strtab[4] + name
            n = elf[a:elf.index(b"\0", a)].decode()
            if n.endswith(".kd") and size == 64 and shndx < shnum:
                d = sec[shndx]
                out[n[:-3]] = struct.unpack_from("<II", elf, d[4] + value - d[3])
    return out


@pytest.fixture(scope="module")
def kernels():
    if not os.path.exists(build.LIB):
        build.build_product()
    with open(build.LIB, "rb") as f:
        data = f.read()
    k = {}
    for elf in _code_objects(data):
        k.update(_descriptors(elf))
    assert any("k_shade" in n for n in k) and any("k_dn_level" in n for n in k) and any("k_lbvh_boxes" in n for n in k)
    return k


def test_render_loop_kernels_use_no_scratch_memory(kernels):
    loop = {n: v[1] for n, v in kernels.items() if re.search(r"\dk_(init|extend|shade|shadow|secondary|resolve|nrc)", n)}
    assert len(loop) > 20 and {n: s for n, s in loop.items() if s} == {}


def test_batched_shade_variants_all_carry_media(kernels):
    feats = [re.search(r"8FeaturesILb(\d)ELb(\d)ELb(\d)ELb(\d)E", n).groups() for n in kernels if "k_shadeILb1E" in n]
    # plain and extended, with and without textures; no radiance cache
    assert sorted(feats) == [("0", "0", "0", "1"), ("0", "0", "1", "1"), ("1", "0", "0", "1"), ("1", "0", "1", "1")]

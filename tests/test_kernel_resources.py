"""Registers that the compiler spilled in kernels that cannot afford it, from the metadata of the built library's code objects."""

import struct

import pytest

msgpack = pytest.importorskip("msgpack")


def _kernels(blob: bytes):
    """The kernels' metadata of every gfx950 code object in the bundles of a library's .hip_fatbin."""
    magic, at = b"__CLANG_OFFLOAD_BUNDLE__", 0
    while (at := blob.find(magic, at)) >= 0:
        n, pos = struct.unpack_from("<Q", blob, at + len(magic))[0], at + len(magic) + 8
        for _ in range(n):
            offset, size, idlen = struct.unpack_from("<QQQ", blob, pos)
            name = blob[pos + 24 : pos + 24 + idlen]
            pos += 24 + idlen
            if b"gfx950" in name and size:
                yield from _notes(blob[at + offset : at + offset + size])
        at += len(magic)


def _notes(elf: bytes):
    shoff, (shentsize, shnum) = struct.unpack_from("<Q", elf, 40)[0], struct.unpack_from("<HH", elf, 58)
    for i in range(shnum):
        kind, _, _, offset, size = struct.unpack_from("<IQQQQ", elf[shoff + i * shentsize + 4 :][:36])
        if kind != 7:  # SHT_NOTE
            continue
        pos = offset
        while pos < offset + size:
            namesz, descsz, _ = struct.unpack_from("<III", elf, pos)
            start = pos + 12 + (namesz + 3) // 4 * 4
            if elf[pos + 12 : pos + 12 + namesz].rstrip(b"\0") == b"AMDGPU":
                yield from msgpack.unpackb(elf[start : start + descsz], strict_map_key=False)["amdhsa.kernels"]
            pos = start + (descsz + 3) // 4 * 4


@pytest.fixture(scope="module")
def kernels():
    from deepseekternarized_amd.kernels import _lib

    if not _lib.LIB_PATH.exists():  # built only when nothing is there
        from deepseekternarized_amd.build import build

        build(verbose=False)
    return list(_kernels(_lib.LIB_PATH.read_bytes()))


# fp16 scales, six loads per loader, one tile per barrier (K = 7168); fp4 kernel with 8 waves and two or four tokens. The launches that
# add to their outputs are one of the two objects of their source: the counts are what these kernels had without the other case.
@pytest.mark.parametrize("name,sgprs,vgprs", [("k_tq1_gemv_cwILi2ELi6ELi1ELi1E", 185, 0), ("k_tq1_gemv_cwILi2ELi6ELi1ELi4E", 216, 10),
                                              ("k_tq1_gemv_fp4ILi2ELi8ELi0ELi2ELi1ELi0E", 24, 0), ("k_tq1_gemv_fp4ILi2ELi8ELi0ELi4ELi1ELi0E", 26, 0)])
def test_streaming_kernels_that_add_spill_no_more(kernels, name, sgprs, vgprs):
    spills = [(k[".sgpr_spill_count"], k[".vgpr_spill_count"]) for k in kernels if name in k[".name"]]
    assert len(spills) == 2
    assert any(s <= sgprs and v <= vgprs for s, v in spills), spills

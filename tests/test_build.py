"""The built library's code objects (host only)."""
import struct

import pytest

PAGE = 4096


def device_functions(lib: bytes):
    """(name, address) of every function in the gfx950 code objects of `lib`:
    clang's offload bundles, each entry an ELF64 file."""
    at = 0
    while (at := lib.find(b"__CLANG_OFFLOAD_BUNDLE__", at)) >= 0:
        count, pos = struct.unpack_from("<Q", lib, at + 24)[0], at + 32
        for _ in range(count):
            off, size, n = struct.unpack_from("<QQQ", lib, pos)
            triple = lib[pos + 24:pos + 24 + n]
            pos += 24 + n
            if b"gfx950" in triple and size:
                yield from elf_functions(lib[at + off:at + off + size])
        at += 24


def elf_functions(elf: bytes):
    assert elf[:4] == b"\x7fELF"
    shoff, = struct.unpack_from("<Q", elf, 40)
    shentsize, shnum = struct.unpack_from("<HH", elf, 58)
    section = lambda i: struct.unpack_from("<IIQQQQIIQQ", elf, shoff + i * shentsize)
    for i in range(shnum):
        _, kind, _, _, off, size, link, _, _, entsize = section(i)
        if kind != 11:  # SHT_DYNSYM
            continue
        names = section(link)[4]
        for s in range(off, off + size, entsize):
            name, info, _, _, value, _ = struct.unpack_from("<IBBHQQ", elf, s)
            if info & 15 == 2:  # STT_FUNC
                yield elf[names + name:elf.index(b"\0", names + name)].decode(), value


def test_kernels_start_on_pages():
    """A kernel's place, and with it the pages that its code touches, does not
    depend on the kernels before it in its file."""
    from rwkv_mlx_amd.build import LIB_PATH
    if not LIB_PATH.exists():
        pytest.skip("not built")
    found = list(device_functions(LIB_PATH.read_bytes()))
    assert len(found) > 100 and any("pipe_kernel" in n for n, _ in found)
    assert [n for n, value in found if value % PAGE] == []

"""No device function of the kernel library is called out of line: a walk's
short stack is passed by reference, and through a real call it lives in memory
and the caller's values in the registers a call preserves (directLight of the
generic kernel: 188-199 VGPRs instead of 157-165, 25 % slower)."""
import struct

from visrtx_amd import _native

BUNDLE = b"__CLANG_OFFLOAD_BUNDLE__"


def _code_objects(data: bytes):
    """The gfx950 code objects of a host library's offload bundles."""
    at = data.find(BUNDLE)
    while at >= 0:
        n, = struct.unpack_from("<Q", data, at + 24)
        p = at + 32
        for _ in range(n):
            off, size, length = struct.unpack_from("<QQQ", data, p)
            triple = data[p + 24:p + 24 + length].decode()
            p += 24 + length
            if "gfx950" in triple:
                yield data[at + off:at + off + size]
        at = data.find(BUNDLE, at + 24)


def _functions(elf: bytes):
    """(names of functions, names of kernels) in a code object's symbol table."""
    shoff, = struct.unpack_from("<Q", elf, 0x28)
    shentsize, shnum = struct.unpack_from("<HH", elf, 0x3A)
    sections = [struct.unpack_from("<IIQQQQIIQQ", elf, shoff + i * shentsize) for i in range(shnum)]
    funcs, kernels = set(), set()
    for s in sections:
        if s[1] != 2:   # SHT_SYMTAB
            continue
        names = sections[s[6]][4]
        for q in range(s[4], s[4] + s[5], s[9]):
            name, info, _, shndx = struct.unpack_from("<IBBH", elf, q)
            text = elf[names + name:elf.index(b"\0", names + name)].decode()
            if info & 15 == 2 and shndx:    # STT_FUNC, defined here
                funcs.add(text)
            elif text.endswith(".kd"):
                kernels.add(text[:-3])
    return funcs, kernels


def test_no_out_of_line_device_functions():
    with open(_native.HIP_LIB_PATH, "rb") as f:
        objs = list(_code_objects(f.read()))
    assert objs
    seen = set()
    for elf in objs:
        funcs, kernels = _functions(elf)
        assert not funcs - kernels, sorted(funcs - kernels)
        seen |= kernels
    assert any("k_render" in k for k in seen) and any("k_render_batch" in k for k in seen)

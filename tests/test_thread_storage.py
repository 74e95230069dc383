"""How the built libraries find their thread-local storage."""
import struct

PT_TLS, SHT_RELA, R_X86_64_TLSDESC, EM_X86_64 = 7, 4, 36, 62


def elf(path):
    blob = open(path, "rb").read()
    phoff, shoff = struct.unpack_from("<QQ", blob, 32)
    phsize, phnum, shsize, shnum = struct.unpack_from("<HHHH", blob, 54)
    machine, = struct.unpack_from("<H", blob, 18)
    segments = {struct.unpack_from("<I", blob, phoff + i * phsize)[0] for i in range(phnum)}
    kinds = set()
    for i in range(shnum):
        kind, = struct.unpack_from("<I", blob, shoff + i * shsize + 4)
        at, size = struct.unpack_from("<QQ", blob, shoff + i * shsize + 24)
        if kind == SHT_RELA:
            kinds |= {struct.unpack_from("<I", blob, at + k + 8)[0] for k in range(0, size, 24)}
    return machine, segments, kinds


def test_no_descriptors(rt):
    """The C library before 2.40 may lose vector registers in a thread's first access through a TLS descriptor."""
    for path in (rt.LIB_PATH, rt.BINDING_PATH):
        machine, _, kinds = elf(path)
        assert machine != EM_X86_64 or R_X86_64_TLSDESC not in kinds, path


def test_the_binding_has_none(rt):
    """It is loaded last: while a thread has not come to its storage, every other library's lookups in that thread take the long way."""
    assert PT_TLS not in elf(rt.BINDING_PATH)[1]

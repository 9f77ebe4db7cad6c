"""CPU tests of what the built kernels ask of a SIMD: the registers a kernel is
given decide how many of its wavefronts run at once."""
import re
import struct
from pathlib import Path

from svfsiplus_amd import _lib, build

MAGIC = b"__CLANG_OFFLOAD_BUNDLE__"


def _code_objects():
    """The device code objects inside the library."""
    _lib.load()
    lib, at = Path(build.LIB).read_bytes(), -1
    while (at := lib.find(MAGIC, at + 1)) >= 0:
        p = at + len(MAGIC) + 8
        for _ in range(struct.unpack_from("<Q", lib, p - 8)[0]):
            off, size, n = struct.unpack_from("<QQQ", lib, p)
            if lib[p + 24:p + 24 + n].startswith(b"hip") and size:
                yield lib[at + off:at + off + size]
            p += 24 + n


def _registers():
    """Kernel name -> vector registers a wavefront is given, from the kernel
    descriptors (the granulated count, in eights, of compute_pgm_rsrc1)."""
    out = {}
    for elf in _code_objects():
        shoff, = struct.unpack_from("<Q", elf, 0x28)
        shent, shnum = struct.unpack_from("<HH", elf, 0x3A)
        sec = [struct.unpack_from("<IIQQQQIIQQ", elf, shoff + shent * k) for k in range(shnum)]
        for s in (s for s in sec if s[1] == 11):  # SHT_DYNSYM
            names = sec[s[6]][4]
            for at in range(s[4], s[4] + s[5], 24):
                st, _, _, shndx, value, size = struct.unpack_from("<IBBHQQ", elf, at)
                name = elf[names + st:elf.index(b"\0", names + st)].decode()
                if name.endswith(".kd") and shndx:
                    rsrc1, = struct.unpack_from("<I", elf, sec[shndx][4] + value - sec[shndx][3] + 48)
                    out[name[:-3]] = 8 * ((rsrc1 & 63) + 1)
    return out


def test_unsplit_dots_run_four_wavefronts():
    """The FP64 dots of large systems (one workgroup for all columns) are kernels
    of their own and run four wavefronts a SIMD; the split form of small systems,
    four columns at a time, has its own registers."""
    r = _registers()
    assert len(r) > 50
    for kind in ("k_mdot", "k_bmdot"):
        got = {n: v for n, v in r.items() if re.match(rf"_ZN3svg\d+{kind}(ILi\d+EE|E)", n)}
        one = [512 // v for n, v in got.items() if "ILi1EE" in n]
        assert len(got) == 2 and one == [4], got

"""Registers and scratch of the transform kernels, read from the built library's kernel descriptors.

The dispatch and the launch bounds count on a number of wavefronts per SIMD,
which a change elsewhere in a kernel can shift without any result changing.
"""
import os
import re
import struct

import pytest

LIB = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "provenloop_amd",
                   "libtensafe_he_hip.so")
PM, INT = "NS_7PmArithE", "NS_8IntArithE"


def _sections(elf):
    shoff, = struct.unpack_from("<Q", elf, 0x28)
    size, count, names = struct.unpack_from("<HHH", elf, 0x3A)
    heads = [struct.unpack_from("<IIQQQQIIQQ", elf, shoff + i * size) for i in range(count)]
    strings = heads[names][4]
    return [(elf[strings + h[0]:elf.index(b"\0", strings + h[0])].decode(), h) for h in heads]


def _kernels(elf):
    """(name, descriptor) of every kernel of an AMD GPU code object."""
    sections = _sections(elf)
    heads = [h for _, h in sections]
    for name, h in sections:
        if name != ".symtab":
            continue
        strings = heads[h[6]][4]
        for off in range(h[4], h[4] + h[5], 24):
            st_name, _, _, shndx, value, size = struct.unpack_from("<IBBHQQ", elf, off)
            sym = elf[strings + st_name:elf.index(b"\0", strings + st_name)].decode()
            if sym.endswith(".kd") and size == 64:
                sec = heads[shndx]
                at = sec[4] + value - sec[3]
                yield sym[:-3], elf[at:at + 64]


@pytest.fixture(scope="module")
def kernels():
    """{mangled name: (wavefronts per SIMD its registers allow, scratch bytes per lane)} of every kernel."""
    if not os.path.exists(LIB):
        pytest.skip("the HIP library is not built")
    lib = open(LIB, "rb").read()
    out = {}
    for m in re.finditer(b"__CLANG_OFFLOAD_BUNDLE__", lib):
        base = m.start()
        count, = struct.unpack_from("<Q", lib, base + 24)
        if count > 16:
            continue  # the magic as a string, not a bundle
        pos = base + 32
        for _ in range(count):
            off, size, idlen = struct.unpack_from("<QQQ", lib, pos)
            target = lib[pos + 24:pos + 24 + idlen]
            pos += 24 + idlen
            if b"gfx950" not in target:
                continue
            for name, kd in _kernels(lib[base + off:base + off + size]):
                scratch, = struct.unpack_from("<I", kd, 4)
                rsrc1, = struct.unpack_from("<I", kd, 48)
                vgprs = 8 * ((rsrc1 & 63) + 1)
                out[name] = (min(8, 512 // vgprs), scratch)
    assert out
    return out


def _find(kernels, pattern):
    found = {n: v for n, v in kernels.items() if re.search(pattern, n)}
    assert found, pattern
    return found


@pytest.mark.parametrize("logn", [13, 14, 15])
def test_large_inverse_passes_keep_their_wavefronts(kernels, logn):
    """On chains of folded primes, launches larger than the caches: row pass four wavefronts per SIMD, column pass
    three; the smaller ones' instances as many as their registers allow."""
    for column, waves in ((0, 4), (1, 3)):
        name = f"16ntt_split_kernelI{PM}Li{logn}ELb1ELb{column}ELj0ELj0ELb"
        assert [w for w, _ in _find(kernels, name + "1E").values()] == [waves]
        assert [w for w, _ in _find(kernels, name + "0E").values()] == [5]


def test_split_kernels_do_not_spill(kernels):
    """None of them, on either arithmetic above 2^41."""
    for name, (_, scratch) in _find(kernels, "ntt_split_kernel|rescale_column_kernel|encrypt_row_kernel|2rd_").items():
        assert scratch == 0, name


@pytest.mark.parametrize("kind,logn,waves", [(PM, 13, 3), (PM, 14, 3), (PM, 15, 3), (INT, 13, 3), (INT, 14, 3), (INT, 15, 2)])
def test_rescale_columns_keep_their_wavefronts(kernels, kind, logn, waves):
    for w, _ in _find(kernels, f"21rescale_column_kernelI{kind}Li{logn}E").values():
        assert w == waves


@pytest.mark.parametrize("kind", [PM, INT])
@pytest.mark.parametrize("logn", [13, 14, 15])
def test_forward_rows_and_encryption_keep_their_wavefronts(kernels, kind, logn):
    """Four per SIMD: the plain forward row pass and the encryption's."""
    for name in (f"16ntt_split_kernelI{kind}Li{logn}ELb0ELb0ELj0ELj0ELb0E", f"18encrypt_row_kernelI{kind}Li{logn}E"):
        for w, _ in _find(kernels, name).values():
            assert w >= 4

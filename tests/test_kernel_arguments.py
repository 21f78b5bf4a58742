"""Kernel arguments of the plain products (no GPU needed: the metadata of the built library).
At 4 us a product of a small sector is its launch, so that a plain product must not carry the
arguments of a Lanczos step."""
import os
import struct

import msgpack
import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
LIB = os.path.join(ROOT, "pyqcm_amd", "libqed.so")


def _code_objects(data):
    magic, at = b"__CLANG_OFFLOAD_BUNDLE__", 0
    while (at := data.find(magic, at)) >= 0:
        n, p = struct.unpack_from("<Q", data, at + 24)[0], at + 32
        for _ in range(n):
            off, size, length = struct.unpack_from("<QQQ", data, p)
            if b"gfx950" in data[p + 24:p + 24 + length] and size:
                yield data[at + off:at + off + size]
            p += 24 + length
        at += len(magic)


def _kernels(elf):
    """The kernel descriptions in the AMDGPU metadata notes (type 32) of a code object."""
    table = struct.unpack_from("<Q", elf, 0x28)[0]
    entry, n = struct.unpack_from("<HH", elf, 0x3A)
    for i in range(n):
        if struct.unpack_from("<I", elf, table + i * entry + 4)[0] != 7:  # SHT_NOTE
            continue
        p, size = struct.unpack_from("<QQ", elf, table + i * entry + 0x18)
        end = p + size
        while p < end:
            name, desc, kind = struct.unpack_from("<III", elf, p)
            d = p + 12 + (name + 3 & ~3)
            if kind == 32:
                yield from msgpack.unpackb(elf[d:d + desc])["amdhsa.kernels"]
            p = d + (desc + 3 & ~3)


def _arguments(kernel):
    """Bytes of the arguments that the host passes (without the runtime's hidden ones)."""
    return max(a[".offset"] + a[".size"] for a in kernel[".args"] if not a[".value_kind"].startswith("hidden"))


@pytest.mark.parametrize("family,plain,step", [("k_hv_ellI", 184, 272), ("k_hv_ell2I", 192, 280),
                                               ("k_hv_ell_batchI", 40, 120), ("k_hv_mixedI", 216, 304),
                                               ("k_hv_generalI", 112, 200)])
def test_plain_products_take_no_lanczos_arguments(family, plain, step):
    if not os.path.exists(LIB):
        pytest.skip("libqed.so not built (run __graft_entry__.build())")
    with open(LIB, "rb") as f:
        found = [k for c in _code_objects(f.read()) for k in _kernels(c) if family in k[".name"]]
    sizes = {True: set(), False: set()}
    for k in found:
        sizes["Step" in k[".name"]].add(_arguments(k))
    assert sizes[False] == {plain} and sizes[True] == {step}, sizes

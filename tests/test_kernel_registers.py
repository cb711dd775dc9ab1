"""CPU tests of what the built library states about its kernels (the metadata notes of its gfx950 code objects): vector
registers spilled to memory, and the registers that decide how many workgroups share a CU."""
import re
import struct

import msgpack
import pytest

from acctransformer_amd import _capi

BUNDLE, ELF_NOTE, AMDGPU_METADATA = b"__CLANG_OFFLOAD_BUNDLE__", 7, 32


def _notes(elf):
    """(type, contents) of the first note of every note section."""
    table, = struct.unpack_from("<Q", elf, 40)
    size, count = struct.unpack_from("<HH", elf, 58)
    for i in range(count):
        kind, = struct.unpack_from("<I", elf, table + i * size + 4)
        at, = struct.unpack_from("<Q", elf, table + i * size + 24)
        if kind == ELF_NOTE:
            name, length, what = struct.unpack_from("<III", elf, at)
            yield what, elf[at + 12 + (name + 3) // 4 * 4:][:length]


@pytest.fixture(scope="module")
def kernels():
    """(kernel, element type, template arguments) -> metadata, of every attention kernel in the library."""
    blob, out = open(_capi.lib_path(), "rb").read(), {}
    for m in re.finditer(BUNDLE, blob):
        count, = struct.unpack_from("<Q", blob, m.start() + 24)
        at = m.start() + 32
        for _ in range(count):
            off, size, name = struct.unpack_from("<QQQ", blob, at)
            target = blob[at + 24:at + 24 + name]
            at += 24 + name
            if b"gfx950" not in target or size == 0:
                continue
            for what, note in _notes(blob[m.start() + off:m.start() + off + size]):
                if what != AMDGPU_METADATA:
                    continue
                for k in msgpack.unpackb(note)["amdhsa.kernels"]:
                    n = re.match(r"_ZN4acct\d+(fa_\w+?_kernel)I(DF16_|DF16b)((?:L[ib]\d+E)*)EEv", k[".name"])
                    if n:
                        out[(n[1], "f16" if n[2] == "DF16_" else "bf16") + tuple(map(int, re.findall(r"L[ib](\d+)E", n[3])))] = k
    return out


def _dkdv(kernels):
    for (name, *key), k in kernels.items():
        if name == "fa_bwd_dkdv_kernel":
            elem, D, bias, drop, mask, ngk = key
            yield (elem, D, bias, drop, ngk), k


def test_every_dkdv_variant_is_seen(kernels):
    assert len(list(_dkdv(kernels))) == 96


def test_no_dkdv_kernel_spills(kernels):
    """A spilled register is reloaded with a wait that also waits for the tile in flight.  (Bias and dropout at head dim 128: two.)"""
    for key, k in _dkdv(kernels):
        elem, D, bias, drop, ngk = key
        assert k[".vgpr_spill_count"] <= (2 if (D, ngk, drop) == (128, 2, 1) and bias else 0), (key, k[".vgpr_spill_count"])


def test_narrow_dkdv_workgroups_share_a_cu(kernels):
    """dkdv_estimate prices one key group per wave at head dims up to 64 as two workgroups of eight waves on a CU: four waves on
    a SIMD, 128 registers each."""
    for key, k in _dkdv(kernels):
        if key[1] <= 64 and key[-1] == 1:
            assert k[".vgpr_count"] <= 128, (key, k[".vgpr_count"])

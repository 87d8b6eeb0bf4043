"""What the built library says without a GPU: register spills of its kernels, from the metadata the compiler leaves in it (a kernel that
touches scratch memory is dispatched more slowly and waits for it in its loop), and a rule that picks kernels by the device's size."""
import ctypes
import importlib
import os
import struct

import pytest

msgpack = pytest.importorskip("msgpack")

LIB = importlib.import_module("turbo-fieldfare_amd").LIB_PATH
NT_AMDGPU_METADATA, SHT_NOTE = 32, 7


def code_objects(raw):
    """The GPU ELF images inside the library's offload bundles."""
    magic, at = b"__CLANG_OFFLOAD_BUNDLE__", 0
    while (at := raw.find(magic, at)) >= 0:
        entry = at + 32
        for _ in range(struct.unpack_from("<Q", raw, at + 24)[0]):
            offset, size, name_len = struct.unpack_from("<QQQ", raw, entry)
            if size and b"gfx950" in raw[entry + 24:entry + 24 + name_len]:
                yield raw[at + offset:at + offset + size]
            entry += 24 + name_len
        at += len(magic)


def kernels():
    with open(LIB, "rb") as f:
        raw = f.read()
    for elf in code_objects(raw):
        sections, (size, count) = struct.unpack_from("<Q", elf, 40)[0], struct.unpack_from("<HH", elf, 58)
        for s in range(sections, sections + size * count, size):
            if struct.unpack_from("<I", elf, s + 4)[0] != SHT_NOTE:
                continue
            note = struct.unpack_from("<Q", elf, s + 24)[0]
            name_len, desc_len, kind = struct.unpack_from("<III", elf, note)
            if kind == NT_AMDGPU_METADATA:
                desc = note + 12 + (name_len + 3) // 4 * 4
                yield from msgpack.unpackb(elf[desc:desc + desc_len])["amdhsa.kernels"]


@pytest.mark.skipif(not os.path.exists(LIB), reason="library not built")
@pytest.mark.parametrize("name", ["qmm_dense_kernel", "qmm_dense_geglu_kernel", "qmm_split_kernel", "grouped_down_mfma_kernel", "attention_prefill_wide_kernel",
                                  "attention_prefill_kernel", "grouped_slice_kernel"])
def test_matrix_core_loops_keep_their_registers(name):
    found = {k[".name"]: k for k in kernels() if f"{len(name)}{name}" in k[".name"]}
    assert found
    assert not {n: k[".vgpr_spill_count"] for n, k in found.items() if k[".vgpr_spill_count"] or k[".private_segment_fixed_size"]}


@pytest.mark.skipif(not os.path.exists(LIB), reason="library not built")
def test_split_tiles_are_chosen_by_the_compute_units_there_are():
    variant = getattr(ctypes.CDLL(LIB), "_ZN3tfk17qmm_split_variantEiiili")      # tfk::qmm_split_variant(m, n, k, ldx, num_cus)
    variant.argtypes, variant.restype = [ctypes.c_int, ctypes.c_int, ctypes.c_int, ctypes.c_long, ctypes.c_int], ctypes.c_int
    none, t32x32, t64x32, t64x64 = range(4)
    tiles = {t32x32: (32, 32), t64x32: (64, 32), t64x64: (64, 64)}
    for cus in (32, 64, 128, 256, 304):
        for m in (1, 32, 33, 64, 65, 128, 200, 500, 1000):
            for n in (64, 2048, 2816, 8192):
                short, got = variant(m, n, 1024, 1024, cus), variant(m, n, 2816, 2816, cus)
                goes = {t: -(-m // rows) * -(-n // cols) / cus for t, (rows, cols) in tiles.items()}
                first = next((t for t in tiles if goes[t] <= 1), t64x64 if m > 64 and goes[t64x64] <= 2 else none)
                assert got == first and short == (none if goes[t64x64] > 1 else first), (cus, m, n)       # two goes only for longer contractions
        assert variant(32, 64, 960, 960, cus) == none and variant(32, 64, 8256, 8256, cus) == none

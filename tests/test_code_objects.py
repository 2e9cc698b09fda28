"""What the compiler made of the kernels (the metadata in the library's own code objects), on the CPU."""
import re
import struct

import pytest

import wgml_amd as W

msgpack = pytest.importorskip("msgpack")


def kernels():
    """name -> metadata of every kernel in the library: its file holds one offload bundle per source file, a bundle the
    ELF file for gfx950, and that a note of type 32 ("AMDGPU") in MessagePack."""
    data = open(W.LIB_PATH, "rb").read()
    found = {}
    for bundle in re.finditer(b"__CLANG_OFFLOAD_BUNDLE__", data):
        at = bundle.end()
        (n,) = struct.unpack_from("<Q", data, at)
        at += 8
        for _ in range(n if n < 16 else 0):
            offset, size, length = struct.unpack_from("<QQQ", data, at)
            target = data[at + 24:at + 24 + length]
            at += 24 + length
            if b"gfx950" not in target or not size:
                continue
            elf = data[bundle.start() + offset:bundle.start() + offset + size]
            (sections,), (entry, count) = struct.unpack_from("<Q", elf, 40), struct.unpack_from("<HH", elf, 58)
            for i in range(count):
                kind, = struct.unpack_from("<I", elf, sections + i * entry + 4)
                start, = struct.unpack_from("<Q", elf, sections + i * entry + 24)
                if kind != 7:  # SHT_NOTE
                    continue
                name_size, desc_size, note = struct.unpack_from("<III", elf, start)
                assert note == 32
                desc = start + 12 + (name_size + 3) // 4 * 4
                for k in msgpack.unpackb(elf[desc:desc + desc_size])["amdhsa.kernels"]:
                    found[k[".name"]] = k
    return found


@pytest.fixture(scope="module")
def all_kernels():
    return kernels()


def test_batched_products_keep_everything_in_registers(all_kernels):
    # (with fewer registers than they need they ran up to 12 % slower than the kernels before them)
    gemm = {n: k for n, k in all_kernels.items() if "gemm_lds_kernel" in n or "gemm_tile_kernel" in n}
    assert len(gemm) == 9 * 2 * 7  # formats, precisions, 16 .. 128 tokens and long runs
    for name, k in gemm.items():
        assert k[".vgpr_spill_count"] == 0 and k[".private_segment_fixed_size"] == 0, name


def test_default_matrix_vector_products_keep_everything_in_registers(all_kernels):
    # (the launch-shape overrides reach the others: two rows per wave or a second tile in flight in Q4_K and Q6_K)
    gemv = {n: k for n, k in all_kernels.items() if "gemv_" in n}
    assert len(gemv) > 150
    spilled = [n for n, k in gemv.items() if k[".vgpr_spill_count"] or k[".private_segment_fixed_size"]]
    for name in spilled:
        assert re.search(r"gemv_quant_i8_kernelINS_7IFmtQ[46]KELi(1ELi[234]|2ELi2)ELi1024E", name), name

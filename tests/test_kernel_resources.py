"""What the compiler made of the kernels, read from the metadata of the built library: arrays that were meant for registers and
went to LDS or scratch memory cost more than the work, and no result shows it."""
import os
import struct

import pytest

msgpack = pytest.importorskip("msgpack")


def _notes(elf: bytes):
    """The code object's metadata map (ELF note of the owner AMDGPU, type 32, msgpack)."""
    shoff, = struct.unpack_from("<Q", elf, 0x28)
    shentsize, shnum = struct.unpack_from("<HH", elf, 0x3A)
    for i in range(shnum):
        kind, = struct.unpack_from("<I", elf, shoff + i * shentsize + 4)
        if kind != 7:  # SHT_NOTE
            continue
        at, size = struct.unpack_from("<QQ", elf, shoff + i * shentsize + 0x18)
        end = at + size
        while at < end:
            name_len, desc_len, kind = struct.unpack_from("<III", elf, at)
            name = elf[at + 12:at + 12 + name_len]
            desc = at + 12 + (name_len + 3) // 4 * 4
            if name.rstrip(b"\0") == b"AMDGPU" and kind == 32:
                return msgpack.unpackb(elf[desc:desc + desc_len], strict_map_key=False)
            at = desc + (desc_len + 3) // 4 * 4
    return None


@pytest.fixture(scope="module")
def kernels():
    from bittorch_amd.build import LIB_PATH
    assert os.path.exists(LIB_PATH), "the library is not built"
    data = open(LIB_PATH, "rb").read()
    magic, found, at = b"__CLANG_OFFLOAD_BUNDLE__", {}, -1
    while (at := data.find(magic, at + 1)) >= 0:
        count, = struct.unpack_from("<Q", data, at + len(magic))
        pos = at + len(magic) + 8
        for _ in range(count if count < 16 else 0):
            offset, size, length = struct.unpack_from("<QQQ", data, pos)
            triple = data[pos + 24:pos + 24 + length]
            pos += 24 + length
            if b"gfx950" in triple and size:
                for k in _notes(data[at + offset:at + offset + size])["amdhsa.kernels"]:
                    found[k[".name"]] = k
    assert found
    return found


def _named(kernels, part):
    got = {n: k for n, k in kernels.items() if part in n}
    assert got, part
    return got.items()


def test_activation_quantizers_keep_their_rows_in_registers(kernels):
    """LDS holds the partial maxima and sums of four waves, nothing else."""
    for name, k in _named(kernels, "act_quant_row_kernel"):
        assert k[".group_segment_fixed_size"] <= 32 and k[".private_segment_fixed_size"] == 0, name
    for name, k in _named(kernels, "act_quant_wave_kernel"):
        assert k[".group_segment_fixed_size"] == 0 and k[".private_segment_fixed_size"] == 0, name


def test_fp32_gemm_waves_work_alone(kernels):
    """Where a wave sums the whole contraction (KS = 1) there is no LDS, and the forward's instances keep everything in registers."""
    for name, k in _named(kernels, "gemm_f32_kernel"):
        src, ks = int(name.split("gemm_f32_kernelILi")[1][0]), int(name.split("ELi")[2][0])
        if ks == 1:
            assert k[".group_segment_fixed_size"] == 0, name
            if src != 2:
                assert k[".private_segment_fixed_size"] == 0 and k[".vgpr_spill_count"] == 0, name

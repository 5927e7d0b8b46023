"""What the compiler records of the built library's kernels: the ones that keep
direct loads in flight across their epilogue spill no vector register (a reload
there waits for every load and store in flight)."""
import struct

import pytest

from hybridagent_amd.build import LIB_PATH

msgpack = pytest.importorskip("msgpack")
MAGIC = b"__CLANG_OFFLOAD_BUNDLE__"


def _code_objects(data):
    at = data.find(MAGIC)
    while at >= 0:
        (n,) = struct.unpack_from("<Q", data, at + len(MAGIC))
        p = at + len(MAGIC) + 8
        for _ in range(n):
            off, size, idlen = struct.unpack_from("<QQQ", data, p)
            name = data[p + 24:p + 24 + idlen]
            p += 24 + idlen
            if b"amdgcn" in name and size:
                yield data[at + off:at + off + size]
        at = data.find(MAGIC, at + len(MAGIC))


def _metadata(elf):
    """The AMDGPU metadata note (type 32) of a 64-bit little-endian ELF."""
    shoff, = struct.unpack_from("<Q", elf, 0x28)
    shentsize, shnum = struct.unpack_from("<HH", elf, 0x3A)
    for i in range(shnum):
        typ, = struct.unpack_from("<I", elf, shoff + i * shentsize + 4)
        off, size = struct.unpack_from("<QQ", elf, shoff + i * shentsize + 0x18)
        while typ == 7 and size >= 12:  # SHT_NOTE
            namesz, descsz, kind = struct.unpack_from("<III", elf, off)
            desc = off + 12 + (namesz + 3) // 4 * 4
            if kind == 32:
                return msgpack.unpackb(elf[desc:desc + descsz])
            step = 12 + (namesz + 3) // 4 * 4 + (descsz + 3) // 4 * 4
            off, size = off + step, size - step
    return {}


@pytest.fixture(scope="module")
def kernels():
    if not LIB_PATH.exists():
        pytest.skip("libw4a16moe.so is not built")
    found = {}
    for obj in _code_objects(LIB_PATH.read_bytes()):
        for k in _metadata(obj).get("amdhsa.kernels", []):
            found[k[".name"]] = k
    assert found, "no kernel metadata in the library"
    return found


@pytest.mark.parametrize("name", ["k_prefill_x", "k_gemm_bf16", "k_linear_w4"])
def test_no_vector_register_spills(kernels, name):
    mine = {n: k for n, k in kernels.items() if name in n}
    assert mine
    spilled = {n: k[".vgpr_spill_count"] for n, k in mine.items()
               if k[".vgpr_spill_count"] or k[".private_segment_fixed_size"]}
    assert not spilled, spilled

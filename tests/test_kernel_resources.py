"""What the compiler made of the kernels, read from the metadata of the built library (no GPU needed): the kernels of the main
path keep everything in registers.  A copy of the parameters or of accumulators in scratch memory costs up to 2.4 times the
time and shows in no result."""
import struct

import pytest

from grouped_mm_bf16_amd import _lib

msgpack = pytest.importorskip("msgpack")


def _code_objects(blob):
    """The device ELFs of every offload bundle in the library."""
    magic, at = b"__CLANG_OFFLOAD_BUNDLE__", 0
    while (at := blob.find(magic, at)) >= 0:
        pos = at + len(magic)
        (count,) = struct.unpack_from("<Q", blob, pos)
        pos += 8
        for _ in range(count):
            offset, size, length = struct.unpack_from("<QQQ", blob, pos)
            name = blob[pos + 24:pos + 24 + length]
            pos += 24 + length
            if b"gfx950" in name and size:
                yield blob[at + offset:at + offset + size]
        at += len(magic)


def _metadata(elf):
    """The kernels' entries in the AMDGPU metadata note."""
    phoff, = struct.unpack_from("<Q", elf, 32)
    phentsize, phnum = struct.unpack_from("<HH", elf, 54)
    for i in range(phnum):
        kind, _, offset, _, _, size = struct.unpack_from("<IIQQQQ", elf, phoff + i * phentsize)
        end = offset + size
        while kind == 4 and offset < end:                     # PT_NOTE
            namesz, descsz, note = struct.unpack_from("<III", elf, offset)
            desc = offset + 12 + (namesz + 3) // 4 * 4
            if note == 32:                                    # NT_AMDGPU_METADATA
                return msgpack.unpackb(elf[desc:desc + descsz], raw=False)["amdhsa.kernels"]
            offset = desc + (descsz + 3) // 4 * 4
    return []


@pytest.fixture(scope="module")
def kernels():
    with open(_lib.LIB_PATH, "rb") as f:
        blob = f.read()
    return {k[".name"]: k for elf in _code_objects(blob) for k in _metadata(elf)}


def test_main_path_uses_no_scratch_memory(kernels):
    staged = {n: k for n, k in kernels.items() if "gmm_staged_kernel" in n}
    asm = {n: k for n, k in kernels.items() if "gmm_asm_kernel" in n}
    assert len(staged) >= 40 and len(asm) >= 20
    scratch = {n: k[".private_segment_fixed_size"] for n, k in {**staged, **asm}.items()}
    fp32 = {n for n in staged if "gmm_staged_kernelIff" in n}
    assert fp32 and {n: s for n, s in scratch.items() if s and n not in fp32} == {}
    # fp32 holds two K tiles in flight and spills a few registers; the parameters (over 200 bytes) must not be among them
    assert {n: scratch[n] for n in fp32 if scratch[n] > 128} == {}

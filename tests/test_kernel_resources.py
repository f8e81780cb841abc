"""Registers of the built kernels, read from the code objects' own metadata: spills and waves per SIMD that a change to shared
code can cost in kernels nobody timed."""
import re
import struct

import msgpack
import pytest

from savanna_amd import _lib


def _code_objects(blob):
    """The gfx950 ELF images of every offload bundle in the library."""
    magic = b"__CLANG_OFFLOAD_BUNDLE__"
    at = blob.find(magic)
    while at >= 0:
        n, = struct.unpack_from("<Q", blob, at + 24)
        p = at + 32
        for _ in range(n):
            off, size, idlen = struct.unpack_from("<QQQ", blob, p)
            if b"gfx950" in blob[p + 24:p + 24 + idlen]:
                yield blob[at + off:at + off + size]
            p += 24 + idlen
        at = blob.find(magic, at + 24)


def _kernels(elf):
    """The metadata maps of an image's kernels (note section, owner AMDGPU, type 32)."""
    shoff, = struct.unpack_from("<Q", elf, 40)
    entsize, num = struct.unpack_from("<HH", elf, 58)
    for i in range(num):
        _, kind, _, _, off, size = struct.unpack_from("<IIQQQQ", elf, shoff + i * entsize)
        end = off + size if kind == 7 else 0
        while off < end:
            namesz, descsz, t = struct.unpack_from("<III", elf, off)
            name = off + 12
            desc = name + (namesz + 3) // 4 * 4
            if t == 32 and elf[name:name + 6] == b"AMDGPU":
                yield from msgpack.unpackb(elf[desc:desc + descsz])["amdhsa.kernels"]
            off = desc + (descsz + 3) // 4 * 4


@pytest.fixture(scope="module")
def kernels():
    blob = open(_lib.LIB_PATH, "rb").read()
    found = {k[".name"]: k for elf in _code_objects(blob) for k in _kernels(elf)}
    assert len(found) > 500
    return found


def _select(kernels, pattern):
    """Kernels by base name and template arguments as they are mangled (int n: Lin, bool: Lb0 / Lb1)."""
    hits = {n: k for n, k in kernels.items() if re.search(pattern, n)}
    assert hits, pattern
    return hits


# Kernels that spill, and how many registers at most.  (The interleaved kernels with a 16-bit featurizer run past the mixer kernels'
# windows only, 16-wave ones in tuning builds only.)
SPILLS = {
    r"toep_bwd_kernelINS_6bf16_tELi5ELi32E": 1,
    r"mfma_il_fwd_kernelINS_(6bf16_t|5f16_t)ELi5ELi16ELi3E": 24,
    r"mfma_il_bwd_kernelINS_6bf16_tELi5ELi8ELb1ELi3E": 4,
    r"mfma_il_bwd_kernelINS_5f16_tELi5ELi8ELb1ELi3E": 12,
    r"dwconv_bwd_kernelINS_(6bf16_t|5f16_t)ELi8ELi8ELb1E": 78,
}


def test_spilled_registers(kernels):
    for pattern in SPILLS:
        _select(kernels, pattern)
    for name, k in kernels.items():
        most = max([n for pattern, n in SPILLS.items() if re.search(pattern, name)], default=0)
        assert k[".vgpr_spill_count"] <= most, (name, k[".vgpr_spill_count"])


# kernel, waves per SIMD that its registers have to leave room for (512 a lane, in eights)
@pytest.mark.parametrize("pattern,waves", [
    (r"mfma_il_fwd_kernelINS_(6bf16_t|5f16_t)ELi5ELi(4|8|16)ELi0E", 4),
    (r"mfma_il_fwd_kernelINS_(6bf16_t|5f16_t)ELi4ELi(8|16)ELi0E", 5),
    (r"mfma_il_fwd_kernelINS_7bf16w_tELi5ELi[48]ELi3E", 2),
    (r"mixer_mr_fwd_kernel", 4),
])
def test_waves_per_simd(kernels, pattern, waves):
    for name, k in _select(kernels, pattern).items():
        vgpr = k[".vgpr_count"]                          # (with the accumulation registers)
        assert 512 // ((vgpr + 7) // 8 * 8) >= waves, (name, vgpr)

"""Registers of the kernels in the built library, from the code objects' own metadata: kernels
whose time hangs on a count of waves per SIMD, or on spilling nothing, keep to it."""

from __future__ import annotations

import re
import struct

import msgpack
import pytest

from zefr_amd import _lib


def _notes(elf):
    """The AMDGPU metadata notes of one 64-bit ELF image."""
    shoff, = struct.unpack_from("<Q", elf, 0x28)
    entsize, num = struct.unpack_from("<HH", elf, 0x3A)
    for i in range(num):
        _, kind, _, _, off, size = struct.unpack_from("<IIQQQQ", elf, shoff + i * entsize)
        end = off + size
        while kind == 7 and off < end:  # SHT_NOTE
            n, d, t = struct.unpack_from("<III", elf, off)
            name = elf[off + 12:off + 12 + n].rstrip(b"\0")
            off += 12 + (n + 3) // 4 * 4
            if name == b"AMDGPU" and t == 32:
                yield msgpack.unpackb(elf[off:off + d], raw=False)
            off += (d + 3) // 4 * 4


def _kernels():
    """{name: metadata} with names like k_divergence<3,9,0,0,1,1> (booleans as 0 and 1)."""
    blob = open(_lib.LIB_PATH, "rb").read()
    out, magic = {}, b"__CLANG_OFFLOAD_BUNDLE__"
    for m in re.finditer(magic, blob):
        at = m.start()
        n, = struct.unpack_from("<Q", blob, at + 24)
        if not 0 < n < 16:
            continue
        pos = at + 32
        for _ in range(n):
            off, size, length = struct.unpack_from("<QQQ", blob, pos)
            triple = blob[pos + 24:pos + 24 + length]
            pos += 24 + length
            if b"gfx950" not in triple:
                continue
            for note in _notes(blob[at + off:at + off + size]):
                for k in note["amdhsa.kernels"]:
                    t = re.match(r"_ZN2zk\d+(k_\w+?)I((?:L[ib]\d+E)+)E", k[".name"])
                    if t:
                        args = re.findall(r"L[ib](\d+)E", t.group(2))
                        out[f"{t.group(1)}<{','.join(args)}>"] = k
    return out


@pytest.fixture(scope="module")
def kernels():
    k = _kernels()
    assert len(k) > 100
    return k


@pytest.mark.parametrize("N", [7, 8, 9])
@pytest.mark.parametrize("flux", [0, 1])
def test_euler_divergence_of_large_hexes_keeps_three_waves(kernels, N, flux):
    """Hexes of order 6 to 8: three waves per SIMD (168 of 512 registers) and no spills, with
    the partner traces extrapolated (SELF) or read."""
    for self_ in (0, 1):
        k = kernels[f"k_divergence<3,{N},0,0,{flux},{self_}>"]
        assert k[".vgpr_count"] <= 168 and k[".vgpr_spill_count"] == 0, (k[".vgpr_count"], k[".vgpr_spill_count"])


@pytest.mark.parametrize("D", [2, 3])
def test_persistent_kernel_scratch(kernels, D):
    """The persistent plan's kernel, a call per phase at three waves per SIMD: its scratch is
    the call frames and a few values (236 and 532 bytes when this was written), which idle
    threads' prologues do not add to."""
    k = kernels[f"k_persist<{D}>"]
    assert k[".private_segment_fixed_size"] <= (240, 540)[D - 2], k[".private_segment_fixed_size"]


@pytest.mark.parametrize("N", range(1, 9))
def test_euler_roe_adjoint_of_quads_keeps_three_waves(kernels, N):
    for form in ("k_adj_main", "k_adj_main_w64"):
        k = kernels[f"{form}<2,{N},0,0,1>"]
        assert k[".vgpr_count"] <= 168 and k[".vgpr_spill_count"] == 0, (k[".vgpr_count"], k[".vgpr_spill_count"])

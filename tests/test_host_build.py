"""The device code in the built library, read from its code objects: no GPU
needed."""

import os
import struct

import msgpack
import numpy as np
import pytest

from wildboar_amd import _lib


@pytest.fixture(scope="module")
def code_objects():
    data = open(_lib.load()._name, "rb").read()
    magic, out, at = b"__CLANG_OFFLOAD_BUNDLE__", [], 0
    while (at := data.find(magic, at)) >= 0:
        (count,) = struct.unpack_from("<Q", data, at + 24)
        entry = at + 32
        for _ in range(count):
            off, size, n = struct.unpack_from("<QQQ", data, entry)
            target = data[entry + 24:entry + 24 + n].decode()
            entry += 24 + n
            if "gfx950" in target and size:
                out.append(data[at + off:at + off + size])
        at += 24
    here = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
    sources = [f for f in os.listdir(os.path.join(here, "wildboar_amd", "csrc"))
               if f.endswith(".hip")]
    assert 0 < len(out) <= len(sources)
    return out


def test_no_scalar_pair_takes_a_literal_for_a_double(code_objects):
    """The compiler sometimes writes a uniform double +inf to a scalar pair as
    s_mov_b64 with a 64-bit literal, which the instruction cannot hold: it is
    encoded with the literal's low half, 0.  (An intended 0 is an inline
    constant.)  rerank.hip starts its threshold in a vector register for that."""
    for elf in code_objects:
        w = np.frombuffer(elf[:len(elf) // 4 * 4], dtype="<u4")
        assert not (((w[:-1] & 0xFF80FFFF) == 0xBE8001FF) & (w[1:] == 0)).any()


def _kernels(elf):
    at = elf.find(b"AMDGPU\0")
    size, kind = struct.unpack_from("<II", elf, at - 8)
    assert kind == 32  # the metadata note: name (8 bytes), then msgpack
    return msgpack.unpackb(elf[at + 8:at + 8 + size])["amdhsa.kernels"]


@pytest.fixture(scope="module")
def registers(code_objects):
    """Vector registers of every kernel, by its mangled name."""
    return {k[".name"]: k[".vgpr_count"] for elf in code_objects for k in _kernels(elf)}


@pytest.mark.parametrize("kernel,most", [
    ("k_lane64_pairsILi8ELi4ELb0ELb0E", 80),   # six waves per SIMD
    ("k_lane64_pairsILi8ELi4ELb1ELb0E", 80),
    ("k_lane64_pairsILi40ELi4ELb1ELb0E", 256),  # two
    ("k_lane_dtwILi40ELi8ELb1ELb0E", 168),     # three
    ("k_lane_dtwILi40ELi8ELb0ELb1E", 160),
])
def test_writing_distances_in_place_keeps_the_waves(registers, kernel, most):
    """The pair kernels' registers leave the waves per SIMD that they have
    without the place of the result kept through the loop."""
    (got,) = [v for name, v in registers.items() if kernel in name]
    assert got <= most


def test_subsequence_scans_do_not_spill(code_objects):
    """The band's offset is a constant of the class, so the tests of which
    window entries lie inside the window are scalar: as wave masks kept over all
    windows they were several hundred spilled registers."""
    spilled = {}
    for elf in code_objects:
        for k in _kernels(elf):
            if "k_subseq_dtw32" in k[".name"]:
                spilled[k[".name"]] = (k[".vgpr_spill_count"], k[".sgpr_spill_count"])
    assert len(spilled) == 32
    assert all(v == 0 and s <= 128 for v, s in spilled.values())

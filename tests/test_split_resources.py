"""Registers of the split kernels, from the metadata of the built library's code
objects: none may spill vector registers, those of K up to 8192 nothing at all
(branches for every form in one kernel once spilled 15 to 58 scalar and up to 16
vector registers, and products of a few hundred rows were 2-7% slower)."""
import re
import shutil
import struct
import subprocess

import pytest

READELF = shutil.which("llvm-readelf") or "/opt/rocm/llvm/bin/llvm-readelf"


def _code_objects(path):
    """The gfx code objects of the offload bundles in a library."""
    data = open(path, "rb").read()
    magic, at = b"__CLANG_OFFLOAD_BUNDLE__", 0
    while (at := data.find(magic, at)) >= 0:
        entries, = struct.unpack_from("<Q", data, at + 24)
        p = at + 32
        for _ in range(entries):
            offset, size, n = struct.unpack_from("<QQQ", data, p)
            name = data[p + 24:p + 24 + n]
            p += 24 + n
            if b"amdgcn" in name and size:
                yield data[at + offset:at + offset + size]
        at += len(magic)


@pytest.fixture(scope="module")
def kernels(tmp_path_factory):
    from ozaki_triton_amd import build
    if not shutil.which(READELF):
        pytest.skip("no llvm-readelf")
    out, tmp = {}, tmp_path_factory.mktemp("co") / "object"
    for obj in _code_objects(build.LIB_PATH):
        tmp.write_bytes(obj)
        notes = subprocess.run([READELF, "--notes", str(tmp)], capture_output=True, text=True).stdout
        for block in notes.split("  - .agpr_count:")[1:]:
            f = dict(re.findall(r"\.(name|sgpr_spill_count|vgpr_spill_count|vgpr_count|"
                                r"private_segment_fixed_size):\s+(\S+)", block))
            out[f["name"]] = tuple(int(f[k]) for k in ("sgpr_spill_count", "vgpr_spill_count",
                                                       "private_segment_fixed_size", "vgpr_count"))
    return out


def test_split_kernels_spill_no_vector_registers(kernels):
    split = {n: r for n, r in kernels.items() if "split_" in n}
    assert len(split) > 100
    assert {n: r for n, r in split.items() if r[1] != 0} == {}


def test_fused_kernels_spill_nothing(kernels):
    """Neither do the kernels of K up to 8192, scalar registers included."""
    fused = {n: r for n, r in kernels.items()
             if "18split_fused_kernel" in n or "17split_rows_kernel" in n}
    assert len(fused) > 100
    assert {n: r for n, r in fused.items() if r[:3] != (0, 0, 0)} == {}


def test_cooperative_column_kernels_fit_three_waves_a_simd(kernels):
    """At most 168 registers: one more leaves two waves, and the fp64 splits took 5-15%
    longer (bf16 slices, whose rounding takes more, have two)."""
    coop = {n: r for n, r in kernels.items()
            if ("17split_pair_kernel" in n or re.search(r"17split_coop_kernel.*Li8EEE", n))
            and "DF16b" not in n}
    assert len(coop) == 12
    assert {n: r for n, r in coop.items() if r[3] > 168} == {}

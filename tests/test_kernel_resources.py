"""Registers of the built library's kernels, where a number decides how many workgroups a compute unit holds."""
import os
import re
import shutil
import subprocess

import pytest

from expertscattergather_amd import _abi

LLVM = "/opt/rocm/llvm/bin"


@pytest.fixture(scope="module")
def kernels(tmp_path_factory):
    """(mangled name, resources) of every kernel in the library's code objects, from their notes."""
    if not _abi.is_built() or not all(os.path.exists(os.path.join(LLVM, tool)) for tool in ("llvm-objdump", "llvm-readelf")):
        pytest.skip("needs the built library and ROCm's llvm tools")
    folder = str(tmp_path_factory.mktemp("code"))
    shutil.copy(_abi.LIB_PATH, os.path.join(folder, "lib.so"))
    subprocess.run([os.path.join(LLVM, "llvm-objdump"), "--offloading", "lib.so"], cwd=folder, check=True, capture_output=True)
    found = []
    for part in sorted(os.listdir(folder)):
        if "gfx950" not in part:
            continue
        notes = subprocess.run([os.path.join(LLVM, "llvm-readelf"), "--notes", part], cwd=folder, check=True, capture_output=True, text=True).stdout
        for block in notes.split("- .agpr_count:")[1:]:
            value = {key: int(re.search(r"\.%s:\s+(\d+)" % key, block).group(1))
                     for key in ("sgpr_count", "vgpr_count", "vgpr_spill_count", "private_segment_fixed_size", "max_flat_workgroup_size")}
            found.append((re.search(r"\.name:\s+(\S+)", block).group(1), value))
    assert len(found) > 500
    return found


def test_two_of_the_routers_workgroups_of_1024_threads_share_a_compute_unit(kernels):
    """Eight wavefronts per SIMD: 80 scalar registers each (16 more are the trap handler's) and, where no row is held, 64 vector registers."""
    large = [(n, k) for n, k in kernels if "router_" in n and k["max_flat_workgroup_size"] == 1024]
    assert len(large) >= 6
    for name, k in large:
        assert k["sgpr_count"] <= 80, (name, k)
        if "ELi0E" in name:                         # the rows' sums from a launch before it
            assert k["vgpr_count"] <= 64, (name, k)


def test_no_kernel_puts_registers_away_in_memory(kernels):
    known = {"_ZN3egs21rows_small_f32_kernelILb1ELi8ELi4ELi2EEEvNS_15SmallRowsParamsE"}      # 128 x 64 weights in registers: four of them, once per tile
    spilled = [(n, k["vgpr_spill_count"], k["private_segment_fixed_size"]) for n, k in kernels if n not in known and (k["vgpr_spill_count"] or k["private_segment_fixed_size"])]
    assert not spilled, spilled


def test_the_fp8_loop_of_32_columns_keeps_two_slabs_ahead(kernels):
    """Two slabs of 64 rows and of 32 columns' weights on their way are 16 + 8 registers, the addresses 24; with fewer than a hundred in all the compiler waits
    for one slab before it asks for the next."""
    (loop,) = [k for n, k in kernels if "tiled_rows_kernelINS_8ElemBF16ELi1ELb1ELi2ELi0E" in n]
    assert loop["vgpr_count"] > 100, loop

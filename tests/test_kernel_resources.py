"""Registers of the built kernels, from the metadata of the library's own gfx950 code objects: none spills to scratch,
and those of D 64 leave room for five waves per SIMD."""
import re
import shutil
import subprocess
from pathlib import Path

import pytest

from gpu_util import no_child_processes_after_gpu_init
from paged_decode import _build

LLVM = Path("/opt/rocm/llvm/bin")


def kernel_notes(tmp_path):
    """(name, VGPRs, spilled VGPRs, spilled SGPRs, scratch bytes) of every kernel of the library."""
    no_child_processes_after_gpu_init()
    for tool in ("llvm-objdump", "llvm-readelf"):
        if not (LLVM / tool).exists():
            pytest.skip(f"{tool} not available")
    library = tmp_path / "lib.so"
    shutil.copy(_build.HIP_LIBRARY, library)
    subprocess.run([LLVM / "llvm-objdump", "--offloading", library], check=True, capture_output=True, cwd=tmp_path)
    kernels = []
    for obj in sorted(tmp_path.glob("lib.so*amdgcn*")):
        notes = subprocess.run([LLVM / "llvm-readelf", "--notes", obj], check=True, capture_output=True, text=True).stdout
        for part in notes.split("- .agpr_count:")[1:]:
            field = {k: int(v) for k, v in re.findall(r"\.(\w+):\s+(\d+)\s", part)}
            kernels.append((re.search(r"\.symbol:\s+'?(\S+?)\.kd", part).group(1), field["vgpr_count"],
                            field["vgpr_spill_count"], field["sgpr_spill_count"], field["private_segment_fixed_size"]))
    return kernels


def test_no_kernel_spills(tmp_path):
    kernels = kernel_notes(tmp_path)
    assert sum("partial_mfma_kernel" in name for name, *_ in kernels) > 100
    assert sum("14partial_kernel" in name for name, *_ in kernels) > 20
    spilled = [k for k in kernels if any(k[2:])]
    assert not spilled, spilled[:8]


def test_d64_kernels_leave_room_for_five_waves_per_simd(tmp_path):
    small = [k for k in kernel_notes(tmp_path) if re.search("partial_mfma_kernel.*Li64ELi", k[0])]
    assert len(small) > 50
    large = [k[:2] for k in small if k[1] > 96]  # 512 VGPRs per SIMD lane, in steps of 8
    assert not large, large[:8]

"""The gather kernels that are held to 64 registers (8 wavefronts per SIMD) keep everything in them: no scratch memory.  Read from the
built library's own metadata, with the tools that built it."""
import glob
import os
import re
import shutil
import subprocess

import pytest

from featgraph_amd import build

TOOLS = "/opt/rocm/llvm/bin"


def _scratch_bytes(tmp_path):
    """Kernel name -> scratch bytes per lane, of every kernel in the library."""
    if not os.path.exists(build.LIB_PATH) or not os.path.exists(os.path.join(TOOLS, "llvm-readelf")):
        pytest.skip("no built library, or no tools to read it with")
    lib = shutil.copy(build.LIB_PATH, tmp_path)
    subprocess.run([os.path.join(TOOLS, "llvm-objdump"), "--offloading", lib], cwd=tmp_path, check=True, stdout=subprocess.DEVNULL)
    found = {}
    for image in glob.glob(os.path.join(tmp_path, "*gfx950")):
        notes = subprocess.run([os.path.join(TOOLS, "llvm-readelf"), "--notes", image], check=True, capture_output=True, text=True).stdout
        for kernel in notes.split(".agpr_count:")[1:]:
            name = re.search(r"\.name:\s+(_Z\S+)", kernel)
            scratch = re.search(r"\.private_segment_fixed_size:\s+(\d+)", kernel)
            found[name.group(1)] = int(scratch.group(1))
    return found


def test_gather_kernels_spill_nothing(tmp_path):
    found = _scratch_bytes(tmp_path)
    for family in ("spmm_items_kernel", "spmm_items_wide_kernel", "spmm_dot_kernel", "attention_items_kernel", "attention_backward_kernel",
                   "additive_sweep_kernel", "sddmm_tiled_kernel", "gspmm_bcast_kernel"):
        kernels = {k: v for k, v in found.items() if family in k}
        assert len(kernels) >= 6, family
        assert {k: v for k, v in kernels.items() if v} == {}, family

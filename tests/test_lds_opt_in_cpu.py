"""Every kernel opts in to more than 64 KiB of LDS for itself.

The launchers remember per kernel and device that it was done. Kernels of one
function type are told apart by a template argument only, so what is checked
here is that the library holds one such record for each kernel of the GEMM
families, where the epilogue's variants share their type.
"""

from __future__ import annotations

import os
import re
import shutil
import subprocess

import pytest

import cuvit_amd


@pytest.mark.skipif(shutil.which("nm") is None, reason="needs nm")
@pytest.mark.parametrize("family", ["gemm_ring_kernel", "gemm_ring_f32_kernel", "gemm_dma_kernel",
                                    "gemm_panel_kernel", "gemm_kernel"])
def test_one_record_per_kernel(family):
    library = os.path.join(os.path.dirname(cuvit_amd.__file__), "..", "lib", "libcuvit_amd.so")
    symbols = subprocess.run(["nm", library], capture_output=True, text=True, check=True).stdout.split()
    name = f"{len(family)}{family}I"  # as the C++ ABI mangles a template's name
    kernels = {s for s in symbols if re.match(rf"_ZN5cuvit6detail4gemm{name}", s)}
    records = {s for s in symbols if "allow_lds" in s and name in s and s.endswith("E7devices")}
    assert kernels
    assert len(records) == len(kernels)

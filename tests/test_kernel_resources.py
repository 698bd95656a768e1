"""Registers that kernels are built with (CPU only: hipcc's resource remarks),
where a wave more or less per SIMD decides the speed of small calls."""
import os
import re
import subprocess

import pytest

from matrix_format_performance_amd import build


@pytest.mark.skipif(not os.path.exists(build.HIPCC), reason="hipcc not present")
def test_csr_vector_row_by_row_keeps_eight_waves():
    r = subprocess.run([build.HIPCC, *build.FLAGS, "--cuda-device-only", "-Rpass-analysis=kernel-resource-usage", "-x",
                        "hip", "-c", os.path.join(build.CSRC, "spmv.hip"), "-o", os.devnull],
                       capture_output=True, text=True, timeout=600)
    assert r.returncode == 0, r.stderr[-2000:]
    waves = re.findall(r"Function Name: _ZN3mfp12k_csr_vectorIfLi(\d+)E.*?Occupancy \[waves/SIMD\]: (\d+)", r.stderr,
                       re.S)
    assert sorted(int(g) for g, _ in waves) == [2, 4, 8, 16, 32, 64]
    assert all(int(w) == 8 for _, w in waves), waves

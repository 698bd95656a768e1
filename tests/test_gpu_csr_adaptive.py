"""CSR-Adaptive row blocks of the sizes whose staged products lie without gaps
in LDS (a CU holds more workgroups so), and FP64 blocks of 16 vectors per lane,
against the oracle's emulator of the summation order, bit for bit."""
import numpy as np
import pytest

import oracle
from gpu_cases import announce

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", ["float32", "float64"])
@pytest.mark.parametrize("W", [1250, 2200, 2600, 4090, 4094, 4095, 4096, 6000, 6300, 8190])
def test_blocks_of_many_entries(gpu, W, dtype):
    announce(f"csr_adaptive W={W} dtype={dtype}")
    rng = np.random.default_rng(W)
    lens = np.concatenate([[W, 1, W - 1, 0, 0, W // 2, W // 2 - 1, 1, 2], rng.integers(0, 70, 4000),
                           np.minimum(1 / (1 - rng.random(3000)), 3000).astype(int), [0] * 700, [W - 3, 2]])
    rp = np.concatenate([[0], np.cumsum(lens)]).astype(np.uint32)
    ci = rng.integers(1, 5003, rp[-1]).astype(np.uint32)
    va = rng.uniform(-1, 1, ci.size).astype(dtype)
    x = gpu.generate_vector(5, 5003, np.dtype(dtype))
    x[0] = np.nan  # read by no entry
    A = gpu.DeviceMatrix.from_csr(rp, ci, va, 5003)
    plan = gpu.Plan(A, "csr_adaptive", nnz_per_wg=W, long_row=16384, chunk=4096)
    xd, yd = gpu.DeviceArray.from_host(x), gpu.DeviceArray(lens.size, np.dtype(dtype))
    yd.fill(np.nan)
    plan.spmv(xd, yd)
    gpu.synchronize()
    assert np.array_equal(yd.to_host(), oracle.spmv_adaptive(rp, ci, va, x, W, 256, 16384, 4096))
    plan.destroy()
    A.destroy()

"""CSR-vector in both of its forms, row by row and from LDS, against the
oracle's emulator of the summation order, bit for bit."""
import numpy as np
import pytest

import oracle
from gpu_cases import announce

pytestmark = pytest.mark.gpu

DTYPES = ["float32", "float64"]


def _csr(lens, cols, dtype, seed=0):
    """Rows of the given lengths with random columns from 1 up (column 0 is
    read by no entry)."""
    rng = np.random.default_rng(seed)
    rp = np.concatenate([[0], np.cumsum(np.asarray(lens, np.int64))]).astype(np.uint32)
    ci = rng.integers(1, cols, rp[-1]).astype(np.uint32)
    return rp, ci, rng.uniform(-1, 1, ci.size).astype(dtype)


# 1.2M and more entries: 9.6 MB in FP32, past the 8 MB from which rows are
# summed from LDS whatever the number of lanes.  Blocks take at most 256 rows.
SHORT = [5, 7] * 100000
ROWS = {
    "chunk edges": SHORT + [1020, 1021, 1023, 1024, 1025, 2044, 2045, 2047, 2048, 2049, 0, 1],
    "every row short": SHORT,
    "rows of 64": [64] * 20001,
}


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("lanes", [2, 8, 64])
@pytest.mark.parametrize("rows", list(ROWS))
def test_rows_of_different_lengths(gpu, rows, lanes, dtype):
    announce(f"csr_vector {rows} lanes={lanes} dtype={dtype}")
    rp, ci, va = _csr(ROWS[rows], 100003, dtype)
    assert ci.size >= 1 << 20
    x = gpu.generate_vector(3, 100003, np.dtype(dtype))
    x[0] = np.nan  # slots past a chunk's elements gather x[0]; none may reach a sum
    A = gpu.DeviceMatrix.from_csr(rp, ci, va, x.size)
    plan = gpu.Plan(A, "csr_vector", lanes=lanes)
    xd, yd = gpu.DeviceArray.from_host(x), gpu.DeviceArray(rp.size - 1, x.dtype)
    yd.fill(np.nan)  # any row left unwritten shows as NaN
    plan.spmv(xd, yd)
    gpu.synchronize()
    assert np.array_equal(yd.to_host(), oracle.spmv_lanes(rp, ci, va, x, lanes))
    plan.destroy()
    A.destroy()

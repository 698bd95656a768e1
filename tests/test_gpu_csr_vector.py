"""CSR-vector over rows of very different lengths: the form that sums rows from
LDS and the blocks of rows that it leaves to their own lanes, against the
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
    "one dense stretch": SHORT[:70001] + [1500] * 300 + SHORT,
    "the first and the last rows": [900] * 130 + SHORT + [700] * 77,
    "sorted by length": sorted(np.minimum(1 / (1 - np.random.default_rng(5).random(160001)), 9000).astype(int))[::-1],
    "chunk edges side by side": SHORT + [1020, 1021, 1023, 1024, 1025, 2044, 2045, 2047, 2048, 2049, 0, 1] * 40,
    "long rows and empty ones": SHORT + [30000, 0, 0, 5000, 0, 2100] * 5 + [0] * 3000,
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


@pytest.mark.parametrize("dtype", DTYPES)
def test_dense_stretch_is_not_one_workgroups_work(gpu, dtype):
    # 256 rows of 1,500 entries side by side among 300,000 short ones, against
    # the same rows spread evenly: in one workgroup they took 47 (FP64: 9)
    # times as long as spread over the chip, by their own lanes 1.5 times
    spread, dense = np.full(300000, 6), np.full(300000, 6)
    spread[::1171][:256] = 1500
    dense[1000:1256] = 1500
    ms = []
    for lens in (spread, dense):
        rp, ci, va = _csr(lens, 300000, dtype)
        announce(f"csr_vector dense stretch dtype={dtype}")
        A = gpu.DeviceMatrix.from_csr(rp, ci, va, 300000)
        plan = gpu.Plan(A, "csr_vector")
        xd = gpu.DeviceArray.from_host(gpu.generate_vector(3, 300000, np.dtype(dtype)))
        yd = gpu.DeviceArray(300000, np.dtype(dtype))
        ms.append(min(sum(plan.kernel_times(xd, yd)) for _ in range(8)))
        plan.destroy()
        A.destroy()
    assert ms[1] < 5 * ms[0], ms

"""COO whose rows are stored by the wave of their first entry: how far past its
span a wave looks depends on the longest row.  Whole numbers, so that every
order of the sums gives the same."""
import numpy as np
import pytest

from gpu_cases import announce

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", ["float32", "float64"])
@pytest.mark.parametrize("longest", [1, 2, 3, 5, 27, 33, 63, 64, 65])
def test_rows_across_spans(gpu, longest, dtype):
    # every row as long as the longest (spans of 256 end inside rows, or with
    # one), then rows of all lengths, the longest among them last
    announce(f"coo rows across spans longest={longest} dtype={dtype}")
    rng = np.random.default_rng(longest)
    lens = np.concatenate([np.full(1200, longest), rng.integers(0, longest + 1, 1500), [longest]])
    rp = np.concatenate([[0], np.cumsum(lens)]).astype(np.uint32)
    ci = rng.integers(0, 5003, rp[-1]).astype(np.uint32)
    va = rng.integers(-3, 4, rp[-1]).astype(dtype)
    x = rng.integers(-5, 6, 5003).astype(dtype)
    A = gpu.DeviceMatrix.from_csr(rp, ci, va, 5003)
    plan = gpu.Plan(A, "coo")
    xd, yd = gpu.DeviceArray.from_host(x), gpu.DeviceArray(lens.size, np.dtype(dtype))
    yd.fill(np.nan)
    plan.spmv(xd, yd)
    gpu.synchronize()
    sums = np.concatenate([[0], np.cumsum(va.astype(np.int64) * x[ci].astype(np.int64))])
    assert np.array_equal(yd.to_host(), (sums[rp[1:]] - sums[rp[:-1]]).astype(dtype))
    plan.destroy()
    A.destroy()

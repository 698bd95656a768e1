"""Kernels chosen by size: each at the sizes where its indexing can go wrong
(chunk and block edges, remainders, empty and very long rows), against the
oracle's emulator of the same summation order, bit for bit, or within the
tolerance of the order-free formats."""
import numpy as np
import pytest

import oracle
from gpu_cases import announce

pytestmark = pytest.mark.gpu

DTYPES = ["float32", "float64"]
RTOL = {np.dtype(np.float32): 1e-5, np.dtype(np.float64): 1e-12}


def _csr(lens, cols, dtype, seed=0):
    """Rows of the given lengths, sorted distinct columns from 1 up (column 0
    is read by no entry)."""
    rng = np.random.default_rng(seed)
    lens = np.asarray(lens, np.int64)
    rp = np.concatenate([[0], np.cumsum(lens)]).astype(np.uint32)
    start = np.repeat(rp[:-1].astype(np.int64), lens)
    t, n = np.arange(rp[-1]) - start, np.repeat(lens, lens)
    lo, hi = t * (cols - 1) // n, (t + 1) * (cols - 1) // n
    ci = 1 + lo + (rng.random(t.size) * (hi - lo)).astype(np.int64)
    return rp, np.minimum(ci, hi).astype(np.uint32), rng.uniform(-1, 1, t.size).astype(dtype)


def _spmv(mfp, rp, ci, va, x, fmt, **tuning):
    announce(f"dispatch fmt={fmt} dtype={va.dtype} rows={rp.size - 1} nnz={ci.size} tuning={tuning}")
    A = mfp.DeviceMatrix.from_csr(rp, ci, va, x.size)
    plan = mfp.Plan(A, fmt, **tuning)
    xd, yd = mfp.DeviceArray.from_host(x), mfp.DeviceArray(rp.size - 1, x.dtype)
    yd.fill(np.nan)  # any row left unwritten shows as NaN
    plan.spmv(xd, yd)
    mfp.synchronize()
    y = yd.to_host()
    plan.destroy()
    A.destroy()
    return y


# A chunk holds 2,048 FP32 (1,024 FP64) elements, less up to 3 (1) where it
# starts off a 16-byte boundary, and 1,984 (960) of a longer row; blocks take
# at most 256 rows.
VECTOR_ROWS = {
    "chunk edges": [1020, 1021, 1022, 1023, 1024, 1025, 2044, 2045, 2046, 2047, 2048, 2049, 0, 1, 2, 3, 959, 960, 961,
                    1983, 1984, 1985] * 2 + [0] * 300 + [90] * 1500,
    "one entry or none": [1, 0] * 140001 + [0] * 255,
    "longest rows": [20011, 0, 0, 7, 39999, 1] * 3 + [64] * 900,
    "a single row": [150001],
    "rows of whole chunks": [8192, 8191, 8193, 4097, 5000] * 5,
}


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("lanes", [2, 16, 64])
@pytest.mark.parametrize("rows", list(VECTOR_ROWS))
def test_csr_vector_from_lds(gpu, rows, lanes, dtype):
    rp, ci, va = _csr(VECTOR_ROWS[rows], 200003, dtype)
    assert ci.size >= 1 << 17  # the size from which the LDS form is chosen
    x = gpu.generate_vector(3, 200003, np.dtype(dtype))
    x[0] = np.nan  # slots past a chunk's elements gather x[0]; none may reach a sum
    y = _spmv(gpu, rp, ci, va, x, "csr_vector", lanes=lanes)
    assert np.array_equal(y, oracle.spmv_lanes(rp, ci, va, x, lanes))


# ---- device memory kept between objects -----------------------------------------

def test_blocks_from_several_threads(gpu):
    # four threads build, multiply and destroy plans of sizes that share
    # memory blocks: none may see another's data
    import threading

    def work(seed, bad):
        gpu.init(0)
        rng = np.random.default_rng(seed)
        for i in range(6):
            rp, ci, va = _csr(rng.integers(0, 40, 9000 + 1500 * int(rng.integers(0, 4))), 9001, "float32", seed + i)
            x = gpu.generate_vector(seed + i, 9001, np.dtype(np.float32))
            y = _spmv(gpu, rp, ci, va, x, "ell" if i % 2 else "csr_scalar")
            if not np.array_equal(y, oracle.spmv_seq(rp, ci, va, x)):
                bad.append((seed, i))

    bad = []
    threads = [threading.Thread(target=work, args=(100 * s, bad)) for s in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not bad


def test_free_memory_counts_kept_blocks(gpu):
    rp, ci, va = _csr([50] * 200000, 200001, "float32")
    free = gpu.device_info()["free_mem"]
    A = gpu.DeviceMatrix.from_csr(rp, ci, va, 200001)
    gpu.Plan(A, "ell").destroy()
    A.destroy()
    assert abs(gpu.device_info()["free_mem"] - free) < 64 << 20

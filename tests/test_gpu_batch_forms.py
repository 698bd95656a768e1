"""Batches at the sizes where the order of their blocks and the forms of their
slices change.  Whole numbers, so that every order of the sums gives the same."""
import numpy as np
import pytest

from gpu_cases import announce

pytestmark = pytest.mark.gpu


def _csr(lens, cols, seed):
    rng = np.random.default_rng(seed)
    rp = np.concatenate([[0], np.cumsum(np.asarray(lens, np.int64))]).astype(np.uint32)
    return rp, np.sort(rng.integers(0, cols, rp[-1])).astype(np.uint32), rng.integers(-3, 4, rp[-1]), cols


def _check(gpu, B, members, k, dtype):
    rng = np.random.default_rng(k)
    X = rng.integers(-5, 6, (B.cols, k))
    Xd, Yd = gpu.DeviceArray.from_host(X.astype(dtype)), gpu.DeviceArray(B.rows * k, np.dtype(dtype))
    Yd.fill(np.nan)
    B.spmm(k, Xd, Yd)
    gpu.synchronize()
    Y = Yd.to_host().reshape(B.rows, k)
    for i, (rp, ci, va, cols) in enumerate(members):
        p = va[:, None] * X[B.col_offsets[i]:B.col_offsets[i + 1]][ci]
        sums = np.concatenate([np.zeros((1, k), np.int64), np.cumsum(p, axis=0)])
        assert np.array_equal(Y[B.row_offsets[i]:B.row_offsets[i + 1]], sums[rp[1:]] - sums[rp[:-1]]), i


# A row of 512 entries is a row block of its own.  X rows of 64 bytes and more:
# turned runs of 16 blocks, 128 a round; narrower ones: one range up to 32
# blocks per CU (8,192 of 256 CUs), then runs of 64.
@pytest.mark.parametrize("blocks", [31, 32, 127, 128, 129, 255, 257, 1025])
@pytest.mark.parametrize("k,dtype", [(16, "float32"), (8, "float64"), (16, "float64")])
def test_stream_wide_rows_of_x(gpu, blocks, k, dtype):
    announce(f"batch stream blocks={blocks} k={k} dtype={dtype}")
    cut = blocks // 3
    members = [_csr([512] * n, 700, n) for n in (cut, blocks - cut)]
    mats = [gpu.DeviceMatrix.from_csr(rp, ci, va.astype(dtype), cols) for rp, ci, va, cols in members]
    B = gpu.Batch(mats, lanes=3)
    _check(gpu, B, members, k, dtype)
    B.destroy()
    for m in mats:
        m.destroy()


@pytest.mark.parametrize("more", [-1, 0, 1])
@pytest.mark.parametrize("k,dtype", [(4, "float32"), (2, "float64")])
def test_stream_narrow_rows_of_x(gpu, more, k, dtype):
    blocks = 32 * gpu.device_info()["cu_count"] + more
    announce(f"batch stream blocks={blocks} k={k} dtype={dtype}")
    members = [_csr([512] * n, 700, n) for n in (blocks - 700, 700)]
    mats = [gpu.DeviceMatrix.from_csr(rp, ci, va.astype(dtype), cols) for rp, ci, va, cols in members]
    B = gpu.Batch(mats, lanes=3)
    _check(gpu, B, members, k, dtype)
    B.destroy()
    for m in mats:
        m.destroy()

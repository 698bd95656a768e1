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


# Column-sorted batches.  Slices with aligned rows (bands) are summed row by row
# from k = 4 in FP32 (there above four items per CU: 1,024 slices of 2,048 rows)
# and k = 8 in FP64 (slices of 1,024 rows from 262,144 rows on; 64 to 16 rows per
# workgroup), where they hold a tenth of the entries.  Members end inside
# slices and inside workgroups.
def _band(rows, width, seed):
    lens = np.full(rows, width)
    lens[5::1013] = 0
    rp = np.concatenate([[0], np.cumsum(lens)]).astype(np.uint32)
    r = np.repeat(np.arange(rows), lens)
    ci = np.minimum(r, rows - width) + np.arange(rp[-1]) - rp[r]
    return rp, ci.astype(np.uint32), np.random.default_rng(seed).integers(-3, 4, ci.size), rows


@pytest.mark.parametrize("k,dtype,rows", [(4, "float32", 1100003), (8, "float32", 150001), (16, "float32", 150001),
                                          (8, "float64", 150001), (16, "float64", 150001), (16, "float32", 9003),
                                          (4, "float64", 150001), (2, "float32", 300007)])
def test_column_sorted_with_aligned_members(gpu, k, dtype, rows):
    announce(f"batch aligned members k={k} dtype={dtype} rows={rows}")
    rng = np.random.default_rng(rows)
    members = [_band(rows, 3, 1), _csr(rng.integers(0, 5, rows // 2 + 77), 5000, 2), _band(rows // 3 + 11, 9, 3),
               _csr(rng.integers(0, 4, rows // 4 + 5), 70001, 4), _band(1037, 128, 5), _band(2053, 129, 6)]
    mats = [gpu.DeviceMatrix.from_csr(rp, ci, va.astype(dtype), cols) for rp, ci, va, cols in members]
    B = gpu.Batch(mats, lanes=1, flags=4, scoo_slice_size=8192, scoo_pieces=1)
    _check(gpu, B, members, k, dtype)
    B.destroy()
    for m in mats:
        m.destroy()


# Slices shrink below 3/4 of a slice per CU (a slice per CU under 2,048 rows),
# to 256 rows at the least.
@pytest.mark.parametrize("dtype", ["float32", "float64"])
@pytest.mark.parametrize("k", [2, 4, 8])
@pytest.mark.parametrize("per_cu", [0.01, 0.74, 0.76, 1.01])
def test_column_sorted_slices_of_few_rows(gpu, per_cu, k, dtype):
    full = {2: 4096, 4: 2048, 8: 1024}[k]  # rows of a slice with half of the LDS
    rows = int(per_cu * gpu.device_info()["cu_count"] * full) + 13
    announce(f"batch few rows k={k} dtype={dtype} rows={rows}")
    rng = np.random.default_rng(rows)
    members = [_csr(rng.integers(0, 4, n), 3001, n) for n in (rows // 3, rows - rows // 3)]
    mats = [gpu.DeviceMatrix.from_csr(rp, ci, va.astype(dtype), cols) for rp, ci, va, cols in members]
    B = gpu.Batch(mats, lanes=1, flags=4, scoo_slice_size=8192, scoo_pieces=1)
    _check(gpu, B, members, k, dtype)
    B.destroy()
    for m in mats:
        m.destroy()

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
# at most 256 rows.  The smaller of these matrices are summed row by row; from 8
# MB of entries see test_gpu_csr_vector.py.
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
# ---- converters ---------------------------------------------------------------
# Tiles of the sort hold 2,048 entries below 2,097,152 of them, then 4,096;
# digits have 1 to 8 bits; tiles of entry rows hold 2,048.

def _triplets(rows, cols, n, seed, dup):
    rng = np.random.default_rng(seed)
    r = rng.integers(0, rows, n).astype(np.uint32)
    c = rng.integers(0, cols, n).astype(np.uint32)
    if dup:  # equal (row, column) pairs keep their input order
        r, c = r // np.uint32(dup) * np.uint32(dup), c // np.uint32(dup) * np.uint32(dup)
    return r, c, rng.uniform(-1, 1, n)


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("rows,cols,n,dup", [
    (1, 1, 1, 0), (1, 1, 3000, 0), (3, 2, 2047, 0), (257, 256, 2048, 0), (256, 257, 2049, 0), (65537, 1, 5000, 0),
    (1, 100000, 6001, 0), (1000003, 1000003, 70001, 0), (4294967295 // 64, 4294967295, 4097, 0),
    (70000, 70000, (1 << 21) - 1, 3), (1023, 5000, 1 << 21, 0), (1024, 100, (1 << 21) + 4097, 0),
    (5, 3000, 70000, 0), (30, 3000, 2200000, 0), (5000, 30000, 300, 7),
    (50000, 50000, (1 << 22) - 1, 50), (50000, 300, 1 << 22, 0), (1 << 20, 1 << 20, (1 << 22) + 8193, 7)])
def test_triplets_any_size(gpu, rows, cols, n, dup, dtype):
    announce(f"triplets rows={rows} cols={cols} n={n} dup={dup} dtype={dtype}")
    r, c, v = _triplets(rows, cols, n, n % 97, dup)
    A = gpu.DeviceMatrix.from_triplets(rows, cols, r, c, v, np.dtype(dtype))
    rp, ci, va = A.download()
    A.destroy()
    order = np.lexsort((c, r))  # stable: ties in input order
    assert np.array_equal(rp, np.searchsorted(r[order], np.arange(rows + 1, dtype=np.int64)).astype(np.uint32))
    assert np.array_equal(ci, c[order])
    assert np.array_equal(va, v[order].astype(dtype))


@pytest.mark.parametrize("where", ["row", "column"])
def test_triplets_out_of_range_are_refused(gpu, where):
    r, c, v = _triplets(1000, 1000, 9001, 3, 0)
    (r if where == "row" else c)[8999] = 1000
    with pytest.raises(gpu.MfpError):
        gpu.DeviceMatrix.from_triplets(1000, 1000, r, c, v)


ENTRY_ROWS = {
    "tile edges": [2047, 1, 0, 2048, 0, 0, 2049, 1, 2046] + [3] * 4000,
    "empty runs": [0] * 40000 + [1] + [0] * 50000 + [1, 2, 3] + [0] * 33000,
    "one row": [5000],
    "all ones": [1] * 4099,
}


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("width", [0, 2])
@pytest.mark.parametrize("rows", list(ENTRY_ROWS))
def test_coo_entries_and_tails(gpu, rows, width, dtype):
    rp, ci, va = _csr(ENTRY_ROWS[rows], 7001, dtype)
    announce(f"coo build {rows} width={width} dtype={dtype}")
    A = gpu.DeviceMatrix.from_csr(rp, ci, va, 7001)
    plan = gpu.Plan(A, "hyb", hyb_width=width) if width else gpu.Plan(A, "coo")
    row = np.repeat(np.arange(rp.size - 1), np.diff(rp.astype(np.int64)))
    tail = np.arange(ci.size) - rp[row] >= width
    from matrix_format_performance_amd import _lib as L
    assert np.array_equal(plan.array(L.MFP_ARR_COO_ROWS, np.uint32), row[tail])
    assert np.array_equal(plan.array(L.MFP_ARR_COO_COLS, np.uint32), ci[tail])
    assert np.array_equal(plan.array(L.MFP_ARR_COO_VALUES, np.dtype(dtype)), va[tail])
    plan.destroy()
    A.destroy()


@pytest.mark.parametrize("values", ["f32", "f64", "bf16"])
@pytest.mark.parametrize("rows", list(ENTRY_ROWS))
def test_column_sorted_build(gpu, rows, values):
    # slices of 256 rows, long-row slices among them: every entry placed once
    rp, ci, va = _csr(ENTRY_ROWS[rows], 7001, "float64" if values == "f64" else "float32")
    va = np.round(va * 64) / 64  # exact in BF16, and their sums exact in FP32
    x = gpu.generate_vector(5, 7001, va.dtype)
    x = np.round(x * 64) / 64
    announce(f"column-sorted build {rows} {values}")
    from matrix_format_performance_amd import _lib as L
    A = gpu.DeviceMatrix.from_csr(rp, ci, va.astype(x.dtype), 7001)
    M = A.convert(values) if values == "bf16" else A
    plan = gpu.Plan(M, "scoo", flags=L.MFP_TUNE_SCOO_COLSORT, scoo_slice_size=256, scoo_pieces=0)
    xd, yd = gpu.DeviceArray.from_host(x), gpu.DeviceArray(rp.size - 1, x.dtype)
    yd.fill(np.nan)
    plan.spmv(xd, yd)
    gpu.synchronize()
    y64, _ = oracle.spmv_f64(rp, ci, va, x)
    assert np.array_equal(yd.to_host().astype(np.float64), y64)
    plan.destroy()
    A.destroy()


# Segments of row blocks hold 4,096 rows (16,384 above 262,144 rows:
# test_gpu_row_blocks.py); a block holds at most W entries (a longer row alone)
# and W + 1 rows.
BLOCK_ROWS = {
    "segment edges": [2] * 16384 * 3,
    "one short of a segment": [3] * 16383,
    "one past a segment": [1] * 16385,
    "empty rows over segments": [0] * 40000 + [5] + [0] * 30000 + [9] * 3 + [0] * 17000,
    "all empty": [0] * 33000,
    "long rows": [700, 1, 0, 699, 513, 512, 511, 1] * 9000,
    "one row": [1],
    "mixed": [int(v) for v in np.minimum(1 / (1 - np.random.default_rng(8).random(70001)), 5000)],
}


@pytest.mark.parametrize("W", [1, 2, 64, 511, 512, 2040, 40000])
@pytest.mark.parametrize("rows", list(BLOCK_ROWS))
def test_row_blocks_any_chain(gpu, rows, W):
    announce(f"row blocks {rows} W={W}")
    rp = np.concatenate([[0], np.cumsum(BLOCK_ROWS[rows])]).astype(np.uint32)
    assert np.array_equal(gpu.fill_row_blocks(rp.size - 1, rp, W), oracle.fill_row_blocks(rp, W))


@pytest.mark.parametrize("rows", list(BLOCK_ROWS))
def test_row_statistics(gpu, rows):
    lens = np.asarray(BLOCK_ROWS[rows], np.int64)
    rp = np.concatenate([[0], np.cumsum(lens)]).astype(np.uint32)
    ci = np.zeros(rp[-1], np.uint32)  # statistics read row lengths only
    A = gpu.DeviceMatrix.from_csr(rp, ci, np.ones(rp[-1], np.float32), 1)
    mn, mx, avg, sd = A.row_stats()
    A.destroy()
    dev = int(((lens - int(lens.sum()) // lens.size) ** 2).sum())
    assert (mn, mx, avg) == (lens.min(), lens.max(), lens.sum() // lens.size)
    assert sd == np.sqrt(np.float64(dev) / lens.size)


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("lens", [[1], [0, 0, 17], [16] * 64, [15, 16, 17, 33] * 49, [0] * 63 + [65] + [1] * 64])
def test_ell_build_tiles(gpu, lens, dtype):
    from matrix_format_performance_amd import _lib as L
    rp, ci, va = _csr(lens, 301, dtype)
    A = gpu.DeviceMatrix.from_csr(rp, ci, va, 301)
    plan = gpu.Plan(A, "ell")
    n, w = len(lens), max(lens)
    ev, ec = np.zeros((w, n), dtype), np.zeros((w, n), np.uint32)
    for r in range(n):
        ev[:lens[r], r], ec[:lens[r], r] = va[rp[r]:rp[r + 1]], ci[rp[r]:rp[r + 1]]
    assert np.array_equal(plan.array(L.MFP_ARR_ELL_VALUES, np.dtype(dtype)), ev.ravel())
    assert np.array_equal(plan.array(L.MFP_ARR_ELL_COLS, np.uint32), ec.ravel())
    plan.destroy()
    A.destroy()


# ---- selector features -------------------------------------------------------------
# The distance bins come from reciprocals up to rows cols = 2^53, from divisions
# above; tiles hold 2,048 entries.

@pytest.mark.parametrize("rows,cols", [(1, 1), (10000, 10000), (4096, 10000), (10000, 40000), (65537, 300007),
                                       (4099, 4294967295), (3000001, 3002399751)])
def test_features_any_shape(gpu, rows, cols):
    from matrix_format_performance_amd import selector
    from oracle import selector as ref
    announce(f"features rows={rows} cols={cols}")
    rng = np.random.default_rng(rows % 1000)
    lens = np.zeros(rows, np.int64)
    used = rng.choice(rows, min(rows, 3000), replace=False)
    lens[used] = rng.integers(1, 1 + min(cols, 9), used.size)
    rp = np.concatenate([[0], np.cumsum(lens)]).astype(np.uint32)
    row = np.repeat(np.arange(rows), lens)
    # half of the columns exactly at multiples of 1e-4 cols from the diagonal
    at = (row * np.float64(cols) / rows).astype(np.int64)
    off = (rng.integers(0, 4096, row.size) * (cols // 10000)) * rng.choice([-1, 1], row.size)
    ci = np.where(rng.random(row.size) < 0.5, at + off, rng.integers(0, cols, row.size)) % cols
    order = np.lexsort((ci, row))
    ci = ci[order].astype(np.uint32)
    A = gpu.DeviceMatrix.from_csr(rp, ci, np.ones(ci.size, np.float32), cols)
    got = selector.features(A)
    A.destroy()
    assert np.array_equal(got, ref.features(rp, ci, rows, cols).astype(np.float32))


# ---- COO and hybrids ------------------------------------------------------------
# A wave takes 256 entries (4 per lane) and looks 64 ahead; rows of at most 64
# entries are stored by the wave of their first entry, longer ones are added.

COO_ROWS = {
    "span edges": [255, 1, 256, 257, 0, 3, 252, 4, 0, 0, 320, 321, 319, 63, 64, 65] * 9,
    "lane edges": [1, 2, 3, 4, 5, 6, 7, 8, 9] * 801,
    "ones and gaps": [1, 0, 0, 1] * 5001,
    "longest owned": [64, 0, 64, 1, 63, 7, 62, 64, 64, 3] * 25,
    "one too long": [65, 3, 0, 64, 64] * 25,
    "last row long": [2] * 127 + [64],
    "empty": [0] * 300,
    "single": [1],
    "very long": [9000, 0, 1] * 3 + [5] * 777,
}


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("fmt", ["coo", "hyb", "hyb_atomic"])
@pytest.mark.parametrize("rows", list(COO_ROWS))
def test_coo_rows_of_any_length(gpu, rows, fmt, dtype):
    rp, ci, va = _csr(COO_ROWS[rows], 10007, dtype)
    x = gpu.generate_vector(3, 10007, np.dtype(dtype))
    if fmt == "coo":
        x[0] = np.inf  # no entry reads column 0 (an ELL part's padding multiplies x[0] by zero)
    y = _spmv(gpu, rp, ci, va, x, fmt, **({} if fmt == "coo" else {"hyb_width": 3}))
    x[0] = 0
    y64, absdot = oracle.spmv_f64(rp, ci, va, x)
    assert not np.isnan(y).any()
    # any order of n products and sums is within n u of sum |a x| (u: unit roundoff)
    bound = (max(COO_ROWS[rows]) + 1) * np.finfo(dtype).eps / 2
    assert oracle.tolerance_check(y, y64, absdot, bound) <= bound


# ---- batch SpMM, slices with aligned rows -----------------------------------------
# Batches of few rows: slices of 256 rows, whose aligned ones (k >= 8) go by 32 or
# 16 rows per workgroup, in chunks of 2,048 (FP64 1,024) entries; rows above 128
# entries keep a slice in the column-sorted form.  Larger slices, and k = 4:
# test_gpu_batch_forms.py.

def _band(rows, width, seed, cols=None, gaps=False):
    """Rows of `width` columns side by side along the diagonal."""
    cols = cols or rows
    lens = np.full(rows, min(width, cols))
    if gaps:
        lens[5::11] = 0
        lens[2000 % rows] = 1
    rp = np.concatenate([[0], np.cumsum(lens)]).astype(np.uint32)
    r = np.repeat(np.arange(rows), lens)
    t = np.arange(rp[-1]) - rp[r]
    ci = (np.minimum(r * cols // rows, cols - min(width, cols)) + t).astype(np.uint32)
    return rp, ci, np.random.default_rng(seed).uniform(-1, 1, ci.size), cols


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("k", [1, 2, 4, 8, 16])
def test_batch_aligned_and_random_slices(gpu, k, dtype):
    announce(f"batch aligned slices k={k} dtype={dtype}")
    members = [_band(2048, 27, 0), _band(5001, 5, 1), _band(1, 1, 2), _band(4097, 128, 3), _band(2100, 129, 4),
               _band(3000, 40, 5, cols=9000), _band(6145, 31, 6, gaps=True)]
    for seed in (7, 8):
        lens = np.random.default_rng(seed).integers(0, 30, 4500)
        members.append((*_csr(lens, 4000, "float64", seed), 4000))
    mats = [gpu.DeviceMatrix.from_csr(rp, ci, va.astype(dtype), cols) for rp, ci, va, cols in members]
    B = gpu.Batch(mats, lanes=1, flags=4, scoo_slice_size=2048, scoo_pieces=1)
    X = gpu.generate_vector(11, B.cols * k, np.dtype(dtype))
    Xd, Yd = gpu.DeviceArray.from_host(X), gpu.DeviceArray(B.rows * k, np.dtype(dtype))
    Yd.fill(np.nan)
    B.spmm(k, Xd, Yd)
    gpu.synchronize()
    Y = Yd.to_host().reshape(B.rows, k)
    for i, (rp, ci, va, cols) in enumerate(members):
        for j in range(k):
            x = X.reshape(B.cols, k)[B.col_offsets[i]:B.col_offsets[i + 1], j].copy()
            y64, absdot = oracle.spmv_f64(rp, ci, va.astype(dtype), x)
            y = Y[B.row_offsets[i]:B.row_offsets[i + 1], j]
            # sums in double, rounded once (FP64: at most 129 roundings of each kind)
            bound = 2 * np.finfo(dtype).eps * (1 if dtype == "float32" else 130)
            assert not np.isnan(y).any()
            assert oracle.tolerance_check(y, y64, absdot, bound) <= bound, (i, j)
    B.destroy()
    for m in mats:
        m.destroy()


# Blocks of a batch go to the XCDs in runs of 64 (512 blocks a round): one
# block per row of 512 entries (stream, and CSR-Adaptive with 512 per
# workgroup; the stream up to 32 blocks per CU in one range: see
# test_gpu_batch_forms.py), and 64 rows of a band for each (column-sorted, k =
# 4).  Whole numbers, so every order gives the same sums.
@pytest.mark.parametrize("blocks", [31, 511, 512, 513, 543, 544, 1061])
@pytest.mark.parametrize("form", ["stream", "rows", "aligned"])
def test_batch_blocks_over_the_xcds(gpu, form, blocks):
    announce(f"batch blocks over the XCDs form={form} blocks={blocks}")
    rng = np.random.default_rng(blocks)
    cut = blocks // 3
    members = []
    for n in (cut, blocks - cut):
        if form == "aligned":
            rp, ci, va, cols = _band(64 * n, 3, n)
        else:
            rp, ci, va = _csr([512] * n, 700, "float32", n)
            cols = 700
        members.append((rp, ci, rng.integers(-3, 4, ci.size).astype("float32"), cols))
    mats = [gpu.DeviceMatrix.from_csr(*m) for m in members]
    k = 1 if form == "rows" else 4
    B = {"stream": lambda: gpu.Batch(mats, lanes=3), "rows": lambda: gpu.Batch(mats, lanes=16, nnz_per_wg=512),
         "aligned": lambda: gpu.Batch(mats, lanes=1, flags=4, scoo_slice_size=2048, scoo_pieces=1)}[form]()
    X = rng.integers(-5, 6, B.cols * k).astype("float32")
    Xd, Yd = gpu.DeviceArray.from_host(X), gpu.DeviceArray(B.rows * k, np.dtype("float32"))
    Yd.fill(np.nan)
    B.spmm(k, Xd, Yd)
    gpu.synchronize()
    Y = Yd.to_host().reshape(B.rows, k)
    for i, (rp, ci, va, cols) in enumerate(members):
        xs = X.reshape(B.cols, k)[B.col_offsets[i]:B.col_offsets[i + 1]].astype(np.float64)
        want = np.add.reduceat(va[:, None] * xs[ci], rp[:-1].astype(np.int64), axis=0)
        assert np.array_equal(Y[B.row_offsets[i]:B.row_offsets[i + 1]], want), i
    B.destroy()
    for m in mats:
        m.destroy()


# Column-sorted items of a batch, k = 1: the plan's order up to one per CU,
# largest first up to 4 (256 threads a workgroup rank them), in runs of 8 above.
# Whole numbers, as above.
@pytest.mark.parametrize("slices", [1, 2, 3, 255, 256, 257, 1023, 1024, 1025, 1060])
def test_batch_column_sorted_items(gpu, slices):
    announce(f"batch column-sorted items slices={slices}")
    rng = np.random.default_rng(slices)
    cut = slices // 2
    members = []
    for n in (cut, slices - cut):
        if n:
            lens = rng.integers(0, 4, 512 * n) * rng.integers(0, 2, n).repeat(512) + 1  # equal and unequal items
            rp, ci, _ = _csr(lens, 1500, "float32", n)
            members.append((rp, ci, rng.integers(-3, 4, ci.size).astype("float32"), 1500))
    mats = [gpu.DeviceMatrix.from_csr(*m) for m in members]
    B = gpu.Batch(mats, lanes=1, flags=4, scoo_slice_size=512, scoo_pieces=1)
    X = rng.integers(-5, 6, B.cols).astype("float32")
    Xd, Yd = gpu.DeviceArray.from_host(X), gpu.DeviceArray(B.rows, np.dtype("float32"))
    Yd.fill(np.nan)
    B.spmm(1, Xd, Yd)
    gpu.synchronize()
    Y = Yd.to_host()
    for i, (rp, ci, va, cols) in enumerate(members):
        xs = X[B.col_offsets[i]:B.col_offsets[i + 1]].astype(np.float64)
        want = np.add.reduceat(va * xs[ci], rp[:-1].astype(np.int64))
        assert np.array_equal(Y[B.row_offsets[i]:B.row_offsets[i + 1]], want), i
    B.destroy()
    for m in mats:
        m.destroy()


# CSR-Adaptive row blocks: a lane sums ceil(W / 256) products, a carried row
# reaches back over up to 255 lanes, the row starts come in 256, 512 and more;
# block and run edges, empty rows, the smallest and largest W.
ADAPTIVE_ROWS = {
    "over many lanes": [2039, 1, 2040, 7, 0, 0, 1021, 1019, 1, 1020, 3, 511, 513, 8, 8, 8, 4, 4, 9] * 3,
    "more rows than 512": [0] * 700 + [3] + [0] * 600 + [5] * 300 + [0] * 255 + [1] * 3000,
    "whole runs": [8] * 255 + [16] * 64 + [64] * 33 + [256] * 9 + [0, 1, 2, 3, 4, 5, 6, 7] * 40,
    "empty": [0] * 1500,
    "one": [1],
}


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("W", [1, 5, 255, 257, 1020, 2040, 8190])
@pytest.mark.parametrize("rows", list(ADAPTIVE_ROWS))
def test_csr_adaptive_row_blocks(gpu, rows, W, dtype):
    rp, ci, va = _csr(ADAPTIVE_ROWS[rows], 5003, dtype)
    x = gpu.generate_vector(5, 5003, np.dtype(dtype))
    x[0] = np.nan  # vectors past a block's elements gather x[0]; none may reach a sum
    y = _spmv(gpu, rp, ci, va, x, "csr_adaptive", nnz_per_wg=W, long_row=4096, chunk=4096)
    assert np.array_equal(y, oracle.spmv_adaptive(rp, ci, va, x, W, 256, 4096, 4096))

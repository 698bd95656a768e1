"""The workloads that performance work on this package is measured on.

A case names one thing that a program does with the package, with its sizes:

``spmv``      one multiplication y = A x with a plan that the program keeps
              (solvers, eigenvalue iterations): any format, FP32 / FP64 /
              BF16 / FP16 values;
``batch``     many matrices assembled once, multiplied by k right-hand sides
              in one call;
``triplets``  assembly: unsorted (row, column, value) triplets in device
              memory to a CSR matrix, as a finite-element code or a reader
              that keeps its data on the GPU does it;
``formats``   the benchmark driver's pass over one new matrix: every format
              is built from CSR and multiplied once;
``select``    the learned format selector on a new matrix: structure features,
              then the network's ranking.

The matrices are the families that the package's benchmark, tests and selector
sweep use: 2D 5-point and 3D 27-point stencils, rows of uniform random length,
and power-law row lengths (floor(1 / U), capped), with the columns of a row
drawn one from each of its equal strata.  They are made here with torch, on
the GPU, from the seed alone.
"""
import math
import random

import numpy as np
import torch

import matrix_format_performance_amd as mfp
from matrix_format_performance_amd import _lib, selector

DEVICE = "cuda:0"
VALUE_BYTES = {"f32": 4, "f64": 8, "bf16": 2, "f16": 2}


def listed():
    return [
        # the smallest call: a 256 x 256 grid's Laplacian, where launches and
        # latency are all there is, in the format that is the reference's best
        # on most small matrices
        {"name": "stencil2d_256_coo_f32", "kind": "spmv", "family": "stencil2d", "n": 256, "format": "coo",
         "values": "f32", "laplace": True},
        # the package's benchmark workload in its tuned form: web-like rows,
        # column-sorted sliced COO
        {"name": "powerlaw_1m_scoo_f32", "kind": "spmv", "family": "powerlaw", "rows": 1 << 20, "nnz_hi": 50000,
         "format": "scoo_colsort", "values": "f32", "slice": 16384, "threads": 1024},
        # the same matrix for a program that tunes nothing and needs FP64 and
        # a fixed summation order
        {"name": "powerlaw_1m_adaptive_f64", "kind": "spmv", "family": "powerlaw", "rows": 1 << 20, "nnz_hi": 50000,
         "format": "csr_adaptive", "values": "f64"},
        # a large structured grid in its best FP32 form
        {"name": "stencil3d_128_ell16_f32", "kind": "spmv", "family": "stencil3d", "n": 128, "format": "ell_packed",
         "values": "f32"},
        # a grid of odd size with BF16 values: the precision study's form
        {"name": "stencil3d_101_ell_bf16", "kind": "spmv", "family": "stencil3d", "n": 101, "format": "ell",
         "values": "bf16"},
        # ragged rows (4 to 64 entries anywhere in the row) in the reference's
        # CSR-vector form
        {"name": "uniform_300k_vector_f32", "kind": "spmv", "family": "uniform", "rows": 300007, "nnz_lo": 4,
         "nnz_hi": 64, "bandwidth": 1.0, "format": "csr_vector", "values": "f32"},
        # the reference's hybrid: short rows in ELL, the long tails in COO
        {"name": "powerlaw_400k_hybrid_f32", "kind": "spmv", "family": "powerlaw", "rows": 400009, "nnz_hi": 10000,
         "format": "hyb_atomic", "values": "f32", "width": 10},
        # many mid-sized matrices at once, 16 and 4 right-hand sides (block
        # methods, several load cases)
        {"name": "batch_64_stream_k16_f32", "kind": "batch", "count": 64, "k": 16, "form": "stream", "values": "f32"},
        {"name": "batch_64_colsort_k4_f32", "kind": "batch", "count": 64, "k": 4, "form": "colsort", "values": "f32"},
        # assembly of a large matrix
        {"name": "triplets_powerlaw_1m_f32", "kind": "triplets", "family": "powerlaw", "rows": 1 << 20,
         "nnz_hi": 50000, "values": "f32"},
        # the driver's and the autotuner's work on one new matrix
        {"name": "formats_uniform_150k_f32", "kind": "formats", "family": "uniform", "rows": 150001, "nnz_lo": 4,
         "nnz_hi": 64, "bandwidth": 1.0, "values": "f32"},
        # the selector's work on one new matrix
        {"name": "select_uniform_300k", "kind": "select", "family": "uniform", "rows": 300007, "nnz_lo": 4,
         "nnz_hi": 64, "bandwidth": 0.1, "values": "f32"},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _draw_matrix(rng, families, scale=1.0):
    family = rng.choice(families)
    if family == "stencil2d":
        return {"family": family, "n": _log_int(rng, 64, 1400 * math.sqrt(scale))}
    if family == "stencil3d":
        return {"family": family, "n": _log_int(rng, 16, 128 * scale ** (1 / 3))}
    if family == "uniform":
        lo = rng.randint(1, 32)
        return {"family": family, "rows": _log_int(rng, 5000, 300000 * scale), "nnz_lo": lo,
                "nnz_hi": rng.randint(lo, 64), "bandwidth": round(math.exp(rng.uniform(math.log(1e-2), 0.0)), 4)}
    rows = _log_int(rng, 10000, (1 << 20) * scale)
    return {"family": family, "rows": rows, "nnz_hi": _log_int(rng, 500, min(50000, rows // 2))}


def draw(rng):
    """One more case of the listed ones' ranges: 64 x 64 to 1400 x 1400 and
    16^3 to 128^3 grids, 5 thousand to a million rows, up to about 12 million
    random or 55 million stencil entries, every format and value type."""
    kind = rng.choices(["spmv", "batch", "triplets", "formats", "select"], [10, 3, 2, 2, 2])[0]
    any_family = ["stencil2d", "stencil3d", "uniform", "powerlaw"]
    if kind == "spmv":
        case = _draw_matrix(rng, any_family)
        stencil = case["family"].startswith("stencil")
        forms = ["csr_vector", "csr_adaptive", "csr_scalar", "coo", "scoo"]
        forms += ["ell", "ell", "ell_packed", "ell_packed"] if stencil else ["scoo_colsort", "scoo_colsort", "hyb",
                                                                              "hyb_atomic", "csr_adaptive"]
        case |= {"kind": kind, "format": rng.choice(forms), "values": rng.choice(["f32", "f64"])}
        if case["format"] in ("csr_vector", "ell", "scoo_colsort", "csr_adaptive") and rng.random() < 0.3:
            case["values"] = rng.choice(["bf16", "f16"])
        if case["format"] == "scoo_colsort":
            case["slice"], case["threads"] = rng.choice([(4096, 512), (8192, 512), (16384, 512), (16384, 1024)])
        if case["format"] in ("hyb", "hyb_atomic"):
            case["width"] = rng.randint(2, 16) if case["family"] == "powerlaw" else rng.randint(case["nnz_lo"],
                                                                                                case["nnz_hi"])
        return case
    if kind == "batch":
        form, k = rng.choice([("stream", 4), ("stream", 8), ("stream", 16), ("colsort", 1), ("colsort", 2),
                              ("colsort", 4), ("colsort", 8), ("lanes", 4), ("adaptive", 1)])
        return {"kind": kind, "count": _log_int(rng, 4, 64), "k": k, "form": form, "values": "f32"}
    if kind == "triplets":
        return {"kind": kind, "values": rng.choice(["f32", "f64"]), **_draw_matrix(rng, any_family, 0.2)}
    if kind == "formats":
        return {"kind": kind, "values": rng.choice(["f32", "f64"]), **_draw_matrix(rng, ["stencil2d", "uniform"], 0.4)}
    return {"kind": kind, "values": "f32", **_draw_matrix(rng, ["uniform", "powerlaw"])}


# ---- matrices ------------------------------------------------------------------

def _rows_of(case):
    return case["n"] ** {"stencil2d": 2, "stencil3d": 3}[case["family"]] if "n" in case else case["rows"]


def _mean_entries(case):
    """Expected entries of the case's matrix (exact for the stencils)."""
    if case["family"] == "stencil2d":
        return 5 * case["n"] ** 2 - 4 * case["n"]
    if case["family"] == "stencil3d":
        return (3 * case["n"] - 2) ** 3
    if case["family"] == "uniform":
        return case["rows"] * (case["nnz_lo"] + case["nnz_hi"]) / 2
    # P(floor(1 / U) >= j) = 1 / j
    return case["rows"] * sum(1.0 / j for j in range(1, case["nnz_hi"] + 1))


def _lengths(case, g):
    """Row lengths: one set for the case, so that every seed has as many
    entries, in an order of the seed's own."""
    rows = case["rows"]
    fixed = torch.Generator(device=DEVICE).manual_seed(rows)
    if case["family"] == "uniform":
        length = torch.randint(case["nnz_lo"], case["nnz_hi"] + 1, (rows,), generator=fixed, device=DEVICE)
    else:
        u = 1.0 - torch.rand(rows, generator=fixed, device=DEVICE, dtype=torch.float64)  # (0, 1]
        length = torch.clamp((1.0 / u).floor(), max=case["nnz_hi"]).to(torch.int64)
    return length[torch.randperm(rows, generator=g, device=DEVICE)]


def _structure(case, g):
    """(row lengths, row of each entry, column of each entry), columns sorted
    within a row."""
    family = case["family"]
    if family.startswith("stencil"):
        n = case["n"]
        dims = 2 if family == "stencil2d" else 3
        r = torch.arange(n ** dims, device=DEVICE)
        at = [(r // n ** d) % n for d in reversed(range(dims))]
        if dims == 2:
            steps = [(-1, 0), (0, -1), (0, 0), (0, 1), (1, 0)]
        else:
            steps = [(a, b, c) for a in (-1, 0, 1) for b in (-1, 0, 1) for c in (-1, 0, 1)]
        cols, ok = [], []
        for step in steps:
            to = [p + s for p, s in zip(at, step)]
            ok.append(torch.stack([(t >= 0) & (t < n) for t in to]).all(0))
            c = to[0]
            for t in to[1:]:
                c = c * n + t
            cols.append(c.to(torch.int32))
        cols, ok = torch.stack(cols, 1), torch.stack(ok, 1)
        length = ok.sum(1)
        return length, torch.repeat_interleave(r, length), cols[ok].to(torch.int64)
    rows = cols = case["rows"]
    length = _lengths(case, g)
    row = torch.repeat_interleave(torch.arange(rows, device=DEVICE), length)
    first = torch.cumsum(length, 0) - length
    t = torch.arange(row.numel(), device=DEVICE) - first[row]
    of = length[row]
    window = torch.clamp(torch.full_like(length, max(1, int(case.get("bandwidth", 1.0) * cols))), min=length)
    start = torch.minimum(torch.clamp(torch.arange(rows, device=DEVICE) - window // 2, min=0), cols - window)
    lo = t * window[row] // of
    hi = (t + 1) * window[row] // of
    u = torch.rand(row.numel(), generator=g, device=DEVICE, dtype=torch.float64)
    return length, row, start[row] + torch.minimum(lo + (u * (hi - lo)).to(torch.int64), hi - 1)


def _matrix(case, seed):
    """{rows, length, row, col, val (float64, rounded to the value type), gen}"""
    g = torch.Generator(device=DEVICE).manual_seed(int(seed) * 7919 + 17)
    length, row, col = _structure(case, g)
    rows = length.numel()
    if case.get("laplace"):
        val = torch.where(row == col, 4.0, -1.0).to(torch.float64)
    elif case["family"] == "stencil3d":
        val = torch.randn(row.numel(), generator=g, device=DEVICE).to(torch.float64)
    else:
        val = (torch.rand(row.numel(), generator=g, device=DEVICE) * 2 - 1).to(torch.float64)
    dt = {"f32": torch.float32, "f64": torch.float64, "bf16": torch.bfloat16, "f16": torch.float16}[case["values"]]
    return {"rows": rows, "length": length, "row": row, "col": col, "plain": val, "val": val.to(dt).to(torch.float64),
            "gen": g}


def _vector(case, n, g):
    dt = torch.float64 if case["values"] == "f64" else torch.float32
    return torch.rand(n, generator=g, device=DEVICE, dtype=dt) * 2 - 1


def _host_csr(case, m):
    """(row_ptr, columns, values) on the host; 16-bit types as FP32, which the
    package then converts."""
    rp = torch.zeros(m["rows"] + 1, dtype=torch.int64, device=DEVICE)
    rp[1:] = torch.cumsum(m["length"], 0)
    dt = torch.float64 if case["values"] == "f64" else torch.float32
    return (rp.to(torch.int32).cpu().numpy().view(np.uint32), m["col"].to(torch.int32).cpu().numpy().view(np.uint32),
            m["plain"].to(dt).cpu().numpy())


def _device_matrix(case, m):
    A = mfp.DeviceMatrix.from_csr(*_host_csr(case, m))
    return A.convert(case["values"]) if case["values"] in ("bf16", "f16") else A


class _Memory:
    """The package's device memory as torch sees it; keeps its owner alive."""

    def __init__(self, owner, ptr, shape, typestr):
        self.owner = owner
        self.__cuda_array_interface__ = {"shape": shape, "typestr": typestr, "data": (ptr, False), "version": 2}


def _tensor(owner, ptr, shape, dtype):
    typestr = {np.dtype(np.float32): "<f4", np.dtype(np.float64): "<f8", np.dtype(np.uint32): "<i4"}[np.dtype(dtype)]
    return torch.as_tensor(_Memory(owner, ptr, shape, typestr), device=DEVICE)


def _vectors(case, cols, rows, g, k=1):
    """x (or X) and y (or Y) in the package's arrays, and y as a tensor."""
    x = mfp.DeviceArray.from_host(_vector(case, cols * k, g).cpu().numpy())
    y = mfp.DeviceArray(rows * k, x.dtype)
    y.fill(0.0)
    return x, y, _tensor(y, y.ptr, (rows, k) if k > 1 else (rows,), x.dtype)


# ---- spmv ----------------------------------------------------------------------

def _plan(A, case, fmt=None):
    """A plan with the options that the case names, or the format's defaults."""
    fmt = fmt or case["format"]
    if fmt == "ell_packed":
        return mfp.Plan(A, "ell", flags=_lib.MFP_TUNE_ELL_PACKED)
    if fmt == "scoo_colsort":
        return mfp.Plan(A, "scoo", flags=_lib.MFP_TUNE_SCOO_COLSORT, scoo_slice_size=case.get("slice", 8192),
                        scoo_threads=case.get("threads", 512), scoo_pieces=0)
    if fmt in ("hyb", "hyb_atomic") and "width" in case:
        return mfp.Plan(A, fmt, hyb_width=case["width"])
    return mfp.Plan(A, fmt)


# ---- batches -------------------------------------------------------------------

def _members(case):
    """The members' sizes, the same for every seed: rows log-uniform in
    [1k, 200k], the four families in turn."""
    rng = random.Random(case["count"])
    out = []
    for i in range(case["count"]):
        rows = _log_int(rng, 1000, 200000)
        family = ("stencil2d", "stencil3d", "uniform", "powerlaw")[i % 4]
        if family == "stencil2d":
            c = {"n": int(math.sqrt(rows))}
        elif family == "stencil3d":
            c = {"n": int(round(rows ** (1 / 3)))}
        elif family == "uniform":
            c = {"rows": rows, "nnz_lo": 4, "nnz_hi": 64}
        else:
            c = {"rows": rows, "nnz_hi": min(rows // 2, 10000)}
        out.append({"family": family, "values": case["values"], **c})
    return out


def _batch(members, case):
    if case["form"] == "stream":
        return mfp.Batch(members, lanes=_lib.MFP_BATCH_STREAM)
    if case["form"] == "colsort":
        return mfp.Batch(members, lanes=1, flags=_lib.MFP_TUNE_SCOO_COLSORT, scoo_slice_size=8192, scoo_pieces=1,
                         scoo_threads=1024)
    return mfp.Batch(members, lanes=16)


# ---- formats -------------------------------------------------------------------

FORMATS = ["csr_scalar", "csr_vector", "csr_adaptive", "ell", "coo", "scoo", "hyb", "hyb_atomic", "scoo_colsort"]


# ---- the interface -------------------------------------------------------------

def prepare(case, seed):
    kind = case["kind"]
    if kind == "batch":
        made = [_matrix(c, seed * 1009 + i) for i, c in enumerate(_members(case))]
        members = [_device_matrix(case, m) for m in made]
        B = _batch(members, case)
        g = torch.Generator(device=DEVICE).manual_seed(int(seed) * 31 + 5)
        x, y, out = _vectors(case, B.cols, B.rows, g, case["k"])
        return {"kind": kind, "batch": B, "k": case["k"], "x": x, "y": y, "out": out}
    m = _matrix(case, seed)
    if kind == "triplets":
        order = torch.randperm(m["row"].numel(), generator=m["gen"], device=DEVICE)
        return {"kind": kind, "rows": m["rows"], "code": {"f32": _lib.MFP_F32, "f64": _lib.MFP_F64}[case["values"]],
                "row": m["row"][order].to(torch.int32), "col": m["col"][order].to(torch.int32),
                "val": m["plain"][order].contiguous()}
    A = _device_matrix(case, m)
    if kind == "select":
        return {"kind": kind, "A": A, "net": selector.Selector.default().net}
    if kind == "formats":
        x = mfp.DeviceArray.from_host(_vector(case, A.cols, m["gen"]).cpu().numpy())
        ys = {f: mfp.DeviceArray(A.rows, x.dtype) for f in FORMATS}
        outs = {f: _tensor(y, y.ptr, (A.rows,), x.dtype) for f, y in ys.items()}
        return {"kind": kind, "A": A, "x": x, "ys": ys, "outs": outs, "case": case}
    x, y, out = _vectors(case, A.cols, A.rows, m["gen"])
    return {"kind": kind, "plan": _plan(A, case), "x": x, "y": y, "out": out}


def run(state):
    kind = state["kind"]
    if kind == "spmv":
        state["plan"].spmv(state["x"], state["y"])
        return state["out"]
    if kind == "batch":
        state["batch"].spmm(state["k"], state["x"], state["y"])
        return state["out"]
    if kind == "triplets":
        h = _lib.C.c_void_p()
        _lib.call("mfp_matrix_from_triplets", _lib.C.byref(h), state["code"], state["rows"], state["rows"],
                  state["row"].numel(), state["row"].data_ptr(), state["col"].data_ptr(), state["val"].data_ptr(), 1,
                  None)
        A = mfp.DeviceMatrix(h)
        return {"row_ptr": _tensor(A, A.row_ptr_ptr, (A.rows + 1,), np.uint32),
                "columns": _tensor(A, A.columns_ptr, (A.nnz,), np.uint32),
                "values": _tensor(A, A.values_ptr, (A.nnz,), A.dtype)}
    if kind == "formats":
        for f, y in state["ys"].items():
            plan = _plan(state["A"], state["case"], f)
            plan.spmv(state["x"], y)
            plan.destroy()
        return state["outs"]
    feats = selector.features(state["A"])
    return {"features": feats, "ranking": state["net"].predict(feats[None, :], bf16=True)}


def work(case):
    kind = case["kind"]
    if kind == "batch":
        nnz = sum(_mean_entries(c) for c in _members(case))
        rows = sum(_rows_of(c) for c in _members(case))
        return {"bytes": nnz * 8 + 4 * rows + 8 * rows * case["k"], "flops": 2 * nnz * case["k"]}
    nnz, rows, vb = _mean_entries(case), _rows_of(case), VALUE_BYTES[case["values"]]
    xb = 8 if case["values"] == "f64" else 4
    if kind == "triplets":
        return {"bytes": nnz * 16 + nnz * (4 + vb) + 4 * rows, "flops": nnz}
    if kind == "select":
        return {"bytes": nnz * 4 + rows * 4, "flops": nnz}
    if kind == "formats":
        # each plan reads the CSR arrays and its multiplication writes y; the
        # six formats that are not CSR also write and read a layout of their own
        csr = nnz * (vb + 4) + 4 * rows
        return {"bytes": len(FORMATS) * (csr + 2 * xb * rows) + 6 * 2 * nnz * (vb + 4), "flops": 2 * nnz * len(FORMATS)}
    # 16-bit column offsets where the form stores them
    cb = 2 if case["format"] == "ell_packed" or (case["format"] == "ell" and vb == 2) else 4
    return {"bytes": nnz * (vb + cb) + rows * (4 + 2 * xb), "flops": 2 * nnz}


# ---- the same in 64 bits -------------------------------------------------------

def _multiply(m, x, k=1):
    """A x in float64; x is (cols,) or (cols, k)."""
    y = torch.zeros((m["rows"], k) if k > 1 else (m["rows"],), dtype=torch.float64, device=DEVICE)
    step = (1 << 25) // k
    for at in range(0, m["row"].numel(), step):
        s = slice(at, at + step)
        v = x[m["col"][s]].to(torch.float64)
        y.index_add_(0, m["row"][s], v * (m["val"][s, None] if k > 1 else m["val"][s]))
    return y


def _features(m):
    rows = cols = m["rows"]
    length, row, col = m["length"].to(torch.float64), m["row"], m["col"]
    nnz = row.numel()
    level = torch.floor(torch.log2(torch.clamp(length, min=1))).to(torch.int64)  # exact: lengths are far below 2^52
    mean = nnz / rows
    std = math.sqrt(max(0.0, float((length * length).sum()) / rows - mean * mean))
    longest, empty = float(length.max()), float((length == 0).sum())
    f = [0.0] * 64
    f[0], f[1], f[2] = math.log2(rows + 1) / 32, math.log2(cols + 1) / 32, math.log2(nnz + 1) / 40
    f[3], f[4] = math.log2(1 + mean) / 16, math.log2(1 + longest) / 16
    f[5], f[6], f[7] = min(std / mean if mean else 0.0, 32.0) / 32, empty / rows, math.log2(1 + std) / 16
    bins = torch.where(length == 0, 0, torch.clamp(level + 1, max=23))
    f[8:32] = (torch.bincount(bins, minlength=24).to(torch.float64) / rows).tolist()
    f[32:48] = (torch.bincount(torch.clamp(level, max=15), weights=length, minlength=16) / nnz).tolist()
    d = (col * rows - row * cols).abs().to(torch.float64) / (float(rows) * cols)
    edges = torch.tensor([1e-4 * 4.0 ** k for k in range(7)], dtype=torch.float64, device=DEVICE)
    f[48:56] = (torch.bincount(torch.bucketize(d, edges, right=True), minlength=8).to(torch.float64) / nnz).tolist()
    f[56] = float(torch.floor(d * 16777216.0).to(torch.int64).sum()) / 16777216.0 / nnz
    f[57] = float((col == row).sum()) / nnz
    end = torch.cumsum(m["length"], 0)
    some = m["length"] > 0
    span = col[end[some] - 1] - col[(end - m["length"])[some]] + 1
    f[58] = float(span.sum()) / max(1, span.numel()) / cols
    f[59] = math.log2(rows * longest / nnz) / 16
    f[60], f[61] = float(length[length > 4096].sum()) / nnz, float(length[length <= 4].sum()) / nnz
    f[62], f[63] = float((length > 64).sum()) / rows, 1.0
    return np.array(f)


def exact(case, seed):
    kind = case["kind"]
    if kind == "batch":
        made = [_matrix(c, seed * 1009 + i) for i, c in enumerate(_members(case))]
        rows, k = sum(m["rows"] for m in made), case["k"]
        g = torch.Generator(device=DEVICE).manual_seed(int(seed) * 31 + 5)
        x = _vector(case, rows * k, g).reshape((rows, k) if k > 1 else (rows,))
        out, at = [], 0
        for m in made:
            out.append(_multiply(m, x[at:at + m["rows"]], k))
            at += m["rows"]
        return torch.cat(out)
    m = _matrix(case, seed)
    if kind == "triplets":
        rp = torch.zeros(m["rows"] + 1, dtype=torch.int64, device=DEVICE)
        rp[1:] = torch.cumsum(m["length"], 0)
        return {"row_ptr": rp, "columns": m["col"], "values": m["val"]}
    if kind == "select":
        return {"features": _features(m), "ranking": None}
    y = _multiply(m, _vector(case, m["rows"], m["gen"]))
    return {f: y for f in FORMATS} if kind == "formats" else y

"""The workloads this library's performance is judged on: CSR SpMV and SpMM the way programs call them.

A case is one matrix (family and sizes), a value type, an operation and the way the caller uses the
library:

  planned     the caller analyses the matrix once and keeps the plan (iterative solvers, graph
              ranking, message passing over a fixed graph): one multiply through it
  following   the plan is kept, but A's values may be overwritten between calls without a word:
              every call checks and, where needed, refreshes the plan, then multiplies
  updated     the values do change before every multiply and the caller says so (Newton and time
              steppers on a fixed mesh)
  planless    nothing is kept: the call itself finds its split points
  transposed  y = A^T x of a matrix seen for the first time: build A^T, multiply
  analysed    the matrix is new in every pass: build a plan, multiply once, drop the plan

Sparsity patterns have the same number of stored elements for every seed, so that the work of a
case is known from the case alone.
"""
import math

import numpy as np
import torch

from library_amd import capi

DTYPES = {"f32": torch.float32, "f64": torch.float64}


def _case(op, matrix, dtype, call, alpha=1.0, beta=0.0, ncols=1, **sizes):
    return dict(op=op, matrix=matrix, dtype=dtype, call=call, alpha=alpha, beta=beta, ncols=ncols, **sizes)


def listed():
    return [
        # the smallest call: a narrow band in one solver step, bound by what a launch costs
        dict(name="spmv_band_small_f64", **_case("spmv", "band", "f64", "planned", rows=1280, half=9)),
        # scattered short rows of equal length (a random sparse operator), single precision, y updated in place
        dict(name="spmv_uniform_f32", **_case("spmv", "uniform", "f32", "planned", 1.5, 0.5, rows=1 << 20, cols=1 << 20, per_row=16)),
        # a graph: power-law row lengths with hub rows of 200000 and a few empty rows, double precision
        dict(name="spmv_zipf_f64", **_case("spmv", "zipf", "f64", "planned", rows=1 << 22, cols=1 << 22, mean=8, expo=2.0, longest=200000)),
        # the largest matrix: a two-dimensional grid operator inside a solver
        dict(name="spmv_stencil5_f64", **_case("spmv", "stencil", "f64", "planned", nx=4096, ny=4096, nz=1)),
        # a three-dimensional grid of odd proportions, caller may change coefficients behind the library's back
        dict(name="spmv_stencil7_follow_f64", **_case("spmv", "stencil", "f64", "following", 1.5, 0.5, nx=200, ny=150, nz=100)),
        # the transposed product of a rectangular power-law matrix met for the first time (an adjoint, a bipartite graph)
        dict(name="spmv_zipf_transposed_f32", **_case("spmv", "zipf", "f32", "transposed", rows=300007, cols=250013, mean=12, expo=2.2, longest=20000)),
        # an unstructured mesh in a bandwidth-reducing order whose coefficients change in every step
        dict(name="spmv_near_updated_f64", **_case("spmv", "near", "f64", "updated", rows=700001, cols=700001, per_row=12, reach=50000)),
        # a fresh matrix in every pass: analysis, one multiply
        dict(name="spmv_uniform_analysed_f64", **_case("spmv", "uniform", "f64", "analysed", rows=300000, cols=400000, per_row=16)),
        # message passing over a power-law graph with 64 features, accumulated into C
        dict(name="spmm_zipf_n64_f32", **_case("spmm", "zipf", "f32", "planned", 1.0, 1.0, 64, rows=1 << 20, cols=1 << 20, mean=16, expo=2.2, longest=50000)),
        # a wide dense band times 64 columns (locally dense operators, windowed attention)
        dict(name="spmm_band_n64_f32", **_case("spmm", "band", "f32", "planned", 1.0, 1.0, 64, rows=1 << 20, half=32)),
        # a block of 8 right-hand sides in a double-precision solver on an unstructured mesh
        dict(name="spmm_near_n8_f64", **_case("spmm", "near", "f64", "planned", 1.0, 0.0, 8, rows=400003, cols=400003, per_row=20, reach=3000)),
        # neighbour sums of 100 features over a sampled graph that is used once
        dict(name="spmm_uniform_n100_planless_f32", **_case("spmm", "uniform", "f32", "planless", 1.0, 0.0, 100, rows=150001, cols=150001, per_row=25)),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """One more case: any family, size, type and use within the ranges of the listed ones."""
    dtype = rng.choice(["f32", "f64"])
    alpha, beta = rng.choice([(1.0, 0.0), (1.5, 0.5), (1.0, 1.0)])
    matrix = rng.choice(["uniform", "zipf", "near", "band", "stencil"])
    if rng.random() < 0.6:
        op, ncols = "spmv", 1
        call = rng.choice(["planned", "planned", "planned", "planned", "following", "updated", "planless", "transposed", "analysed"])
        most = 4_000_000 if call in ("transposed", "analysed") else 1 << 25  # stored elements
        rows_most = 1 << 22
    else:
        op, ncols = "spmm", _log(rng, 2, 256)
        call = rng.choice(["planned", "planned", "planned", "planless"])
        most = min(1 << 24, (1 << 29) // ncols)
        rows_most = min(1 << 20, (1 << 25) // ncols)
    if call == "transposed":
        alpha, beta = 1.0, 0.0
    if matrix == "stencil":
        dims = rng.choice([2, 3])
        points = _log(rng, 2000, min(most // (2 * dims + 1), rows_most * 2 if op == "spmv" else rows_most))
        side = max(8, int(points ** (1.0 / dims)))
        nx = max(4, int(side * rng.uniform(0.6, 1.0)))
        ny = max(4, int(side * rng.uniform(0.6, 1.0)))
        sizes = dict(nx=nx, ny=ny, nz=max(4, int(side * rng.uniform(0.6, 1.0))) if dims == 3 else 1)
    elif matrix == "band":
        half = _log(rng, 1, 32)
        sizes = dict(rows=_log(rng, 1000, min(rows_most, most // (2 * half + 1))), half=half)
    else:
        mean = _log(rng, 3, 64)
        rows = _log(rng, 1000, min(rows_most, most // mean))
        cols = max(256, int(rows * rng.choice([1.0, 1.0, rng.uniform(0.3, 2.0)])))
        sizes = dict(rows=rows, cols=cols)
        if matrix == "zipf":
            sizes.update(mean=mean, expo=round(rng.uniform(1.8, 2.6), 2), longest=min(cols, _log(rng, 500, 200000)))
        elif matrix == "near":
            reach = _log(rng, 100, 100000)
            sizes.update(per_row=mean, reach=min(reach, cols // 2 - 1))
        else:
            sizes.update(per_row=mean)
    return _case(op, matrix, dtype, call, alpha, beta, ncols, **sizes)


# ---------------------------------------------------------------------------------- matrices
def _zipf_lengths(c):
    """Row lengths of a power law with the case's mean and longest row, longest first, one row in a
    hundred empty: quantiles of the distribution, the same for every seed."""
    m, p, longest = c["rows"], 1.0 / (c["expo"] - 1.0), float(c["longest"])
    scale = 1.0
    for _ in range(60):  # scale * E[min(u^-p, longest / scale)] = mean
        cap = max(longest / scale, 1.0)
        u0 = cap ** (-1.0 / p)
        tail = math.log(1.0 / u0) if abs(p - 1.0) < 1e-9 else (1.0 - u0 ** (1.0 - p)) / (1.0 - p)
        scale = c["mean"] / (cap * u0 + tail)
    u = (np.arange(m, dtype=np.float64) + 0.5) / m
    lens = np.clip(np.round(scale * u ** -p), 1, longest).astype(np.int64)
    lens[99::100] = 0
    return lens


def _shape(c):
    """rows, columns and stored elements of the case's matrix."""
    if c["matrix"] == "stencil":
        nx, ny, nz = c["nx"], c["ny"], c["nz"]
        m = nx * ny * nz
        nnz = m + 2 * ((nx - 1) * ny * nz + nx * (ny - 1) * nz + nx * ny * (nz - 1))
        return m, m, nnz
    if c["matrix"] == "band":
        m, h = c["rows"], c["half"]
        return m, m, m * (2 * h + 1) - h * (h + 1)
    if c["matrix"] == "zipf":
        return c["rows"], c["cols"], int(_zipf_lengths(c).sum())
    return c["rows"], c["cols"], c["rows"] * c["per_row"]


def _from_table(cols, keep):
    """Row offsets and columns of a matrix given as a table (rows x at most k) of sorted columns."""
    row_ptr = torch.zeros(cols.shape[0] + 1, dtype=torch.int32, device="cuda")
    row_ptr[1:] = torch.cumsum(keep.sum(1), 0)
    return row_ptr, cols[keep].to(torch.int32)


def _scattered(lens, lo, span, gen):
    """Row r holds lens[r] distinct sorted columns, spread over lo[r] .. lo[r] + span - 1."""
    m = lens.numel()
    row_ptr = torch.zeros(m + 1, dtype=torch.int64, device="cuda")
    row_ptr[1:] = torch.cumsum(lens, 0)
    nnz = int(row_ptr[-1])
    row = torch.repeat_interleave(torch.arange(m, device="cuda"), lens, output_size=nnz)
    room = (span - lens + 1)[row].double()  # a sorted sample of 0 .. room - 1 plus 0, 1, 2, ... is sorted and distinct
    key = (torch.rand(nnz, device="cuda", generator=gen, dtype=torch.float64) * room).long()
    key = torch.sort((row << 32) | key)[0] & 0xFFFFFFFF
    col = key + torch.arange(nnz, device="cuda") - row_ptr[row] + lo[row]
    return row_ptr.to(torch.int32), col.to(torch.int32)


def _matrix(c, gen):
    """Row offsets, columns and values on the GPU."""
    m, n, nnz = _shape(c)
    dtype = DTYPES[c["dtype"]]
    if c["matrix"] == "stencil":
        nx, ny, nz = c["nx"], c["ny"], c["nz"]
        i = torch.arange(m, device="cuda", dtype=torch.int32)
        ix, iy, iz = i % nx, (i // nx) % ny, i // (nx * ny)
        near = [(-1, iy > 0, nx), (-1, ix > 0, 1), (1, ix < nx - 1, 1), (1, iy < ny - 1, nx)]
        if nz > 1:
            near = [(-1, iz > 0, nx * ny)] + near + [(1, iz < nz - 1, nx * ny)]
        half = len(near) // 2
        cols = torch.stack([i + d * s for d, _, s in near[:half]] + [i] + [i + d * s for d, _, s in near[half:]], 1)
        keep = torch.stack([k for _, k, _ in near[:half]] + [i >= 0] + [k for _, k, _ in near[half:]], 1)
        row_ptr, col = _from_table(cols, keep)
        # varying coefficients: a diffusion operator, diagonal against its neighbours
        val = -0.5 - torch.rand(nnz, device="cuda", generator=gen, dtype=dtype)
        own = torch.zeros_like(keep)
        own[:, half] = True
        val[own[keep]] = 2.0 * len(near) + torch.rand(m, device="cuda", generator=gen, dtype=dtype)
        return row_ptr, col, val
    if c["matrix"] == "band":
        off = torch.arange(-c["half"], c["half"] + 1, device="cuda", dtype=torch.int32)
        cols = torch.arange(m, device="cuda", dtype=torch.int32)[:, None] + off[None, :]
        row_ptr, col = _from_table(cols, (cols >= 0) & (cols < n))
    else:
        lo, span = torch.zeros(m, dtype=torch.int64, device="cuda"), n
        if c["matrix"] == "zipf":
            lens = torch.from_numpy(_zipf_lengths(c)).cuda()[torch.randperm(m, device="cuda", generator=gen)]
        else:
            lens = torch.full((m,), c["per_row"], dtype=torch.int64, device="cuda")
        if c["matrix"] == "near":
            span = max(2 * c["reach"] + 1, c["per_row"])
            lo = (torch.arange(m, device="cuda") * n // m - c["reach"]).clamp(0, n - span)
        row_ptr, col = _scattered(lens, lo, span, gen)
    val = torch.rand(nnz, device="cuda", generator=gen, dtype=dtype) * 2 - 1
    return row_ptr, col, val


# ---------------------------------------------------------------------------------- measuring
def prepare(case, seed):
    gen = torch.Generator(device="cuda")
    gen.manual_seed(int(seed))
    m, n, nnz = _shape(case)
    dtype, ncols, call = DTYPES[case["dtype"]], case["ncols"], case["call"]
    row_ptr, col, val = _matrix(case, gen)
    rows_in, rows_out = (m, n) if call == "transposed" else (n, m)
    x = torch.rand(rows_in * ncols, device="cuda", generator=gen, dtype=dtype)
    if case["matrix"] != "stencil":
        x = x * 2 - 1
    y = torch.rand(rows_out * ncols, device="cuda", generator=gen, dtype=dtype) * 2 - 1
    spmm = case["op"] == "spmm"
    plan = workspace = None
    if call in ("planned", "following", "updated"):
        plan = capi.Plan(spmm, capi.SPMM_DEFAULT if spmm else capi.SPMV_DEFAULT, dtype, m, n, nnz, row_ptr, ncols=ncols, col=col,
                         val=val, checked=call == "following")
        workspace = torch.empty(max(plan.workspace_bytes, 256), dtype=torch.uint8, device="cuda")
    elif call == "planless":
        vt = capi.value_type(dtype)
        need = (capi.lib().asx_spmm_workspace_bytes(capi.SPMM_DEFAULT, vt, m, nnz, ncols) if spmm
                else capi.lib().asx_spmv_workspace_bytes(capi.SPMV_DEFAULT, vt, m, nnz))
        workspace = torch.empty(max(need, 256), dtype=torch.uint8, device="cuda")
    return dict(case=case, a=(row_ptr, col, val), x=x, y=y, m=m, n=n, nnz=nnz, dtype=dtype, plan=plan, workspace=workspace)


def run(state):
    c, (row_ptr, col, val), x, y = state["case"], state["a"], state["x"], state["y"]
    alpha, beta, call, plan = c["alpha"], c["beta"], c["call"], state["plan"]
    if c["op"] == "spmm":
        return capi.spmm(row_ptr, col, val, x, y, c["ncols"], alpha, beta, plan=plan, workspace=state["workspace"])
    if call == "transposed":
        at = capi.csr_transpose(row_ptr, col, val, state["n"])
        return at + (capi.spmv(*at, x, y, alpha, beta),)
    if call == "analysed":
        plan = capi.Plan(False, capi.SPMV_DEFAULT, state["dtype"], state["m"], state["n"], state["nnz"], row_ptr, col=col, val=val)
        capi.spmv(row_ptr, col, val, x, y, alpha, beta, plan=plan)
        plan.destroy()
        return y
    if call == "following":
        plan.refresh_if_changed(val)
    elif call == "updated":
        plan.update_values(val)
    return capi.spmv(row_ptr, col, val, x, y, alpha, beta, plan=plan, workspace=state["workspace"])


def work(case):
    """A read once, x (B) read once, y (C) written once and, with beta, read once; A^T written once where it is a result."""
    m, n, nnz = _shape(case)
    sv, ncols = (8 if case["dtype"] == "f64" else 4), case["ncols"]
    rows_out = n if case["call"] == "transposed" else m
    nbytes = nnz * (sv + 4) + (m + 1) * 4 + (m + n) * ncols * sv
    if case["beta"] != 0.0:
        nbytes += rows_out * ncols * sv
    if case["call"] == "transposed":
        nbytes += nnz * (sv + 4) + (n + 1) * 4
    return {"bytes": nbytes, "flops": 2 * nnz * ncols}


def tolerance(case):
    """Sums of a row's products in another order; indices and copied values are exact."""
    return {"rel": 1e-5} if case["dtype"] == "f32" else {"rel": 1e-13}

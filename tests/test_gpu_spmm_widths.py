"""The SpMM kernels at the edges of their dispatch: widths of C on both sides of every lane group and column tile,
row lengths around what one lane group takes alone, segment sizes, padded leading dimensions.  Against the CPU oracle;
tolerance: a row's products in another order, tol * (|alpha| sum |a b| + |beta c|) with tol = 1e-12 (fp64), 1e-5 (fp32)."""
import numpy as np
import pytest
import scipy.sparse as sp
import torch

from conftest import csr_from_lengths
from library_amd import capi, workloads as W

pytestmark = pytest.mark.gpu
TOL = {np.dtype(np.float64): 1e-12, np.dtype(np.float32): 1e-5}


def _check(oracle, rp, col, val, k, n, ldb, ldc, beta, planned, what, alg=capi.SPMM_MERGE):
    rng = np.random.default_rng(n)
    m, dtype = rp.size - 1, val.dtype
    B = rng.uniform(-1, 1, (k - 1) * ldb + n).astype(dtype)   # ends with the last column of the last row
    C0 = rng.uniform(-1, 1, (m - 1) * ldc + n).astype(dtype)
    d = [torch.from_numpy(a).cuda() for a in (rp, col, val, B, C0)]
    plan = capi.Plan(True, alg, dtype, m, k, col.size, d[0], ncols=n, col=d[1], val=d[2]) if planned else None
    capi.spmm(d[0], d[1], d[2], d[3], d[4], n, 1.5, beta, alg=alg, plan=plan, ldb=ldb, ldc=ldc, k=k)
    torch.cuda.synchronize()
    got = d[4].cpu().numpy()
    ref = oracle.spmm(rp, col, val, B, n, 1.5, beta, C0, 8, ldb=ldb, ldc=ldc)
    full = lambda a, rows, ld: np.concatenate([a, np.zeros(ld - n, a.dtype)]).reshape(rows, ld)
    scale = 1.5 * (sp.csr_matrix((np.abs(val.astype(np.float64)), col, rp), shape=(m, k)) @ np.abs(full(B, k, ldb)[:, :n].astype(np.float64)))
    scale += abs(beta) * np.abs(full(C0, m, ldc)[:, :n])
    g, r, c0 = full(got, m, ldc), full(ref, m, ldc), full(C0, m, ldc)
    assert np.all(np.abs(g[:, :n] - r[:, :n]) <= TOL[np.dtype(dtype)] * scale), what
    assert np.array_equal(g[:, n:], c0[:, n:]), f"{what}: wrote between the rows of C"
    if plan is not None:
        plan.destroy()


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("n", [1, 2, 3, 4, 5, 8, 9, 16, 17, 32, 33, 64, 65, 127, 128, 129, 255, 256, 257, 515])
def test_spmm_merge_widths(oracle, dtype, n):
    rng = np.random.default_rng(5)
    # rows around what a lane group takes alone (16, 32, 64), empty rows, one that covers segments, a segment of nothing but row ends
    lens = np.r_[rng.integers(0, 12, 200), 15, 16, 17, 31, 32, 33, 63, 64, 65, 0, 0, 1500, np.zeros(300, int), rng.integers(60, 200, 20), 1]
    rp, col, val = csr_from_lengths(lens, 1700, 9, dtype)
    for ldb, ldc, beta, planned in ((n, n, 0.0, False), (n + 1, n + 3, 0.5, True)):
        _check(oracle, rp, col, val, 1700, n, ldb, ldc, beta, planned, f"n={n} ldb={ldb} beta={beta}")


@pytest.mark.parametrize("dtype,m,n", [(np.float32, 70001, 8), (np.float64, 70001, 6), (np.float32, 140001, 36), (np.float32, 140001, 5)])
def test_spmm_merge_segment_sizes(oracle, dtype, m, n):
    """Sizes past which a wave takes 256 and 512 merge items instead of 128."""
    rp, col, val = W.csr_fixed(m, 50000, 16, dtype, seed=3)
    for planned in (False, True):
        _check(oracle, rp, col, val, 50000, n, n, n, 1.0, planned, f"m={m} n={n} planned={planned}")


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("n", [1, 5, 16, 17, 31, 33, 63, 65, 66, 127, 129, 130, 193, 257])
def test_spmm_blocked_widths(oracle, dtype, n):
    """The blocked kernel at the edges of its column tiles, with and without spare columns behind the rows, k no multiple of 4."""
    rng = np.random.default_rng(6)
    m, k = 83, 61
    A = sp.random(m, k, density=0.3, random_state=7, format="csr", dtype=dtype)
    A[40:60] = 0  # block rows without blocks
    A.eliminate_zeros()
    rp, col, val = A.indptr.astype(np.int32), A.indices.astype(np.int32), A.data.astype(dtype)
    for ldb, ldc, beta in ((n, n, 0.0), (n, n, 1.0), (n + 1, n + 3, 0.5)):
        _check(oracle, rp, col, val, k, n, ldb, ldc, beta, True, f"blocked n={n} ldb={ldb} beta={beta}", alg=capi.SPMM_BLOCKED)


@pytest.mark.parametrize("dtype,n", [(np.float64, 1048561), (np.float32, 2097220)])
def test_spmm_merge_most_columns(oracle, dtype, n):
    """More columns than 65535 tiles of 128 bytes hold, rows of B on lines."""
    rp, col, val = csr_from_lengths(np.array([2, 0, 3]), 4, 9, dtype)
    ld = (n + 31) // 32 * 32
    for planned in (False, True):
        _check(oracle, rp, col, val, 4, n, ld, ld, 0.5, planned, f"n={n} planned={planned}")

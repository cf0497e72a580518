"""Kernels whose tiles wait for their stored elements before they gather (grids of more than 2048 workgroups) and the same
kernels on grids that do not: the last tile holds one element, a few, all but one or all, rows are cut and whole, and the last
tiles may hold empty rows only.  Sums of small integers, exact in both types and in any order, against the oracle's."""
import numpy as np
import pytest
import torch

from conftest import row_ptr_from_lengths
from library_amd import capi

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("tiles,last", [(3, 1), (2048, 1024), (2049, 1), (2049, 5), (2050, 1023), (4100, 1024)])
def test_last_tile(oracle, tiles, last, dtype):
    nnz, n = (tiles - 1) * 1024 + last, 5003
    rng = np.random.default_rng(tiles)
    lens = np.minimum(rng.integers(0, 40, nnz // 16), 38)
    lens = lens[: np.searchsorted(np.cumsum(lens), nnz)]
    lens = np.r_[lens, nnz - lens.sum(), np.zeros(3000, int)]
    rp = row_ptr_from_lengths(lens)
    col = rng.integers(0, n, nnz).astype(np.int32)
    val, x, y0 = (rng.integers(-4, 5, k).astype(dtype) for k in (nnz, n, lens.size))
    d = [torch.from_numpy(a).cuda() for a in (rp, col, val, x)]
    ref = oracle.spmv(rp, col, val, x, 2.0, 0.5, y0, 1)
    for alg in (capi.SPMV_STREAM, capi.SPMV_FLAT, capi.SPMV_MERGE, None):
        plan = None if alg is None else capi.Plan(False, alg, val.dtype, lens.size, n, nnz, d[0])
        y = torch.from_numpy(y0).cuda()
        capi.spmv(*d, y, 2.0, 0.5, plan=plan)
        assert np.array_equal(y.cpu().numpy(), ref), alg
        if plan is not None:
            plan.destroy()

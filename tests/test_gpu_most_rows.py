"""Searches over as many rows as an int32 counts: their first step and the last rows' numbers reach 2^31 - 1.  Integers in
float32, so that every order of the sums gives the same bits."""
import numpy as np
import pytest
import torch

from library_amd import capi

pytestmark = pytest.mark.gpu

M, N, TAIL = 2**31 - 1, 1000, 4096


@pytest.fixture(scope="module")
def matrix():
    """One element in every 2048th row, and one more in each of the last 4096."""
    row_ptr = torch.empty(M + 1, dtype=torch.int32, device="cuda")
    step = 1 << 28
    for a in range(0, M + 1, step):
        row_ptr[a:a + step] = torch.arange(a, min(a + step, M + 1), dtype=torch.int64, device="cuda") >> 11
    row_ptr[M - TAIL:] += torch.arange(TAIL + 1, dtype=torch.int32, device="cuda")
    rows = np.sort(np.r_[((np.arange(M >> 11, dtype=np.int64) + 1) << 11) - 1, np.arange(M - TAIL, M)], kind="stable")
    rng = np.random.default_rng(5)
    col = rng.integers(0, N, rows.size).astype(np.int32)
    col[1:][(rows[1:] == rows[:-1]) & (col[1:] == col[:-1])] = 7
    val, x = rng.integers(1, 5, rows.size).astype(np.float32), rng.integers(1, 5, N).astype(np.float32)
    yield row_ptr, rows, col, val, x
    torch.cuda.empty_cache()


def check(matrix, y):
    _, rows, col, val, x = matrix
    held, first = np.unique(rows, return_index=True)
    expect = np.add.reduceat(val * x[col], first)
    assert torch.equal(y[torch.from_numpy(held).cuda()].cpu(), torch.from_numpy(expect))
    assert int(torch.count_nonzero(y)) == held.size


@pytest.mark.parametrize("alg", [None, capi.SPMV_DEFAULT, capi.SPMV_FLAT, capi.SPMV_MERGE])
def test_multiply(matrix, alg):
    """Without a plan (the flat kernel looks its rows up itself), and with plans, whose analysis looks rows up for a sample."""
    row_ptr, rows, col, val, x = matrix
    d = [torch.from_numpy(a).cuda() for a in (col, val, x)]
    y = torch.zeros(M, device="cuda")
    plan = None if alg is None else capi.Plan(False, alg, val.dtype, M, N, rows.size, row_ptr, col=d[0], val=d[1])
    capi.spmv(row_ptr, *d, y, 1.0, 0.0, alg=capi.SPMV_FLAT if alg is None else alg, plan=plan)
    torch.cuda.synchronize()
    if plan is not None:
        plan.destroy()
    check(matrix, y)


def test_transpose(matrix):
    """The wave that holds the last elements marks the starts of rows up to the last one."""
    row_ptr, rows, col, val, _ = matrix
    got = capi.csr_transpose(row_ptr, *[torch.from_numpy(a).cuda() for a in (col, val)], N)
    torch.cuda.synchronize()
    order = np.argsort(col, kind="stable")
    assert np.array_equal(got[0].cpu().numpy(), np.r_[0, np.cumsum(np.bincount(col, minlength=N))])
    assert np.array_equal(got[1].cpu().numpy(), rows[order].astype(np.int32))
    assert np.array_equal(got[2].cpu().numpy(), val[order])

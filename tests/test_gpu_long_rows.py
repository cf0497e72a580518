"""SpMV plans that list their long rows, at the edges of the list: row lengths on both sides of eight turns of a lane group,
of what takes a workgroup and of the longest row the list is for; every lane group.  Against float64 sums on the host;
tolerance: a row's products in another order, len u (|alpha| sum |a x|) + 3 u |beta y| with u = 2^-24 or 2^-53."""
import numpy as np
import pytest
import torch

from conftest import csr_from_lengths
from library_amd import capi

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("lanes", [2, 4, 8, 16, 32])
@pytest.mark.parametrize("wide", [(), (2047, 2048, 2049), (8191, 8192)])
def test_long_row_list(dtype, lanes, wide):
    rng = np.random.default_rng(lanes)
    cut = 8 * lanes
    n = 9001
    short = rng.integers(0, 2 * lanes - 2, 3001)
    lens = np.r_[short[:1500], cut - 1, cut, cut + 1, 0, wide, cut, 1900, short[1500:]].astype(int)
    while lens.sum() > lanes * lens.size:  # keep the mean row inside the lane group
        lens = np.r_[lens, np.ones(1000, int)]
    rp, col, val = csr_from_lengths(lens, n, 3, dtype)
    x, y0 = rng.uniform(-1, 1, n).astype(dtype), rng.uniform(-1, 1, lens.size).astype(dtype)
    d = [torch.from_numpy(a).cuda() for a in (rp, col, val, x)]
    plan = capi.Plan(False, capi.SPMV_DEFAULT, val.dtype, lens.size, n, col.size, d[0], col=d[1], val=d[2])
    assert plan.alg == capi.SPMV_VECTOR
    u = 2.0 ** (-53 if dtype == np.float64 else -24)
    rows = np.repeat(np.arange(lens.size), lens)
    prod = val.astype(np.longdouble) * x[col].astype(np.longdouble)
    exact, size = np.zeros(lens.size, np.longdouble), np.zeros(lens.size, np.longdouble)
    np.add.at(exact, rows, prod)
    np.add.at(size, rows, np.abs(prod))
    for beta in (0.0, 0.5):
        y = torch.from_numpy(y0).cuda()
        capi.spmv(d[0], d[1], d[2], d[3], y, 1.5, beta, plan=plan)
        torch.cuda.synchronize()
        bound = (lens + 3) * u * 1.5 * size + 3 * u * np.abs(beta * y0)
        assert np.all(np.abs(y.cpu().numpy() - (1.5 * exact + beta * y0)) <= bound), (lanes, beta)
    plan.destroy()


def test_one_row_of_every_element_int32_offsets_can_count():
    """2^31 - 1 ones: 64 lanes with two sums each add 2^24 of them at most, exact in float32; joined they round to 2^31."""
    nnz = 2**31 - 1
    row_ptr = torch.tensor([0, nnz], dtype=torch.int32, device="cuda")
    col = torch.zeros(nnz, dtype=torch.int32, device="cuda")
    val = torch.ones(nnz, dtype=torch.float32, device="cuda")
    x, y = torch.ones(1, device="cuda"), torch.full((1,), -7.0, device="cuda")
    capi.spmv(row_ptr, col, val, x, y, 1.0, 0.0, alg=capi.SPMV_VECTOR)
    torch.cuda.synchronize()
    assert y.item() == 2.0**31


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("rows, length, longest, n", [(1, 0, 1000000, 1200000), (1, 0, 30000, 40000), (3, 9000, 9000, 10000),
                                                      (20, 100000, 100000, 200000), (64, 30000, 30000, 100000),
                                                      (1800, 500, 1000000, 1200000), (2, 300000, 2000000, 2500000)])
def test_default_cuts_very_long_rows(dtype, rows, length, longest, n):
    """Few rows, or one among shorter ones, that a single workgroup would walk alone: DEFAULT, with the columns at hand, takes a
    kernel that cuts rows between workgroups.  Integers, so that every order of the sums gives the same bits."""
    rng = np.random.default_rng(rows)
    lens = np.r_[np.full(rows, length, int), longest]
    rp = np.r_[0, np.cumsum(lens)].astype(np.int32)
    col = np.concatenate([np.sort(rng.choice(n, k, replace=False)) for k in lens]).astype(np.int32)
    val, x = rng.integers(-2, 3, col.size).astype(dtype), rng.integers(-2, 3, n).astype(dtype)
    d = [torch.from_numpy(a).cuda() for a in (rp, col, val, x)]
    plan = capi.Plan(False, capi.SPMV_DEFAULT, val.dtype, lens.size, n, col.size, d[0], col=d[1], val=d[2])
    assert plan.alg in (capi.SPMV_FLAT, capi.SPMV_MERGE, capi.SPMV_SLICED, capi.SPMV_WINDOW), plan.alg
    y = torch.zeros(lens.size, dtype=d[2].dtype, device="cuda")
    capi.spmv(*d, y, 1.0, 0.0, plan=plan)
    torch.cuda.synchronize()
    prod = val.astype(np.float64) * x[col]
    expect = [prod[a:b].sum() for a, b in zip(rp[:-1], rp[1:])]
    assert np.array_equal(y.cpu().numpy(), np.array(expect, dtype))
    plan.destroy()

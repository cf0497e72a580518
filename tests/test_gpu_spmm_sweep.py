"""The SpMM kernel whose waves go through the columns of A together: every number of lanes a row of B takes, one and two tiles of
columns, rows a group from one to all it has registers for, rows of uneven length (what a wave stages at once among them), and
calls that stay with the other kernels.  Products of small integers, whose sums are exact in both types and in any order, against
integer sums."""
import numpy as np
import pytest
import torch

from library_amd import capi

pytestmark = pytest.mark.gpu


def _matrix(lens, n, seed, ascending=True):
    """Row offsets, columns (distinct within a row and spread over all n) and values."""
    gen = torch.Generator(device="cuda").manual_seed(seed)
    lens = torch.as_tensor(lens, device="cuda", dtype=torch.int64)
    rp = torch.zeros(lens.numel() + 1, dtype=torch.int64, device="cuda")
    rp[1:] = torch.cumsum(lens, 0)
    row = torch.repeat_interleave(torch.arange(lens.numel(), device="cuda"), lens)
    key = (torch.rand(row.numel(), device="cuda", generator=gen, dtype=torch.float64) * (n - lens + 1)[row]).long()
    col = torch.sort((row << 32) | key)[0] & 0xFFFFFFFF
    col += torch.arange(row.numel(), device="cuda") - rp[row]
    if not ascending:
        col = col[torch.argsort((row << 32) | torch.randint(0, 1 << 30, col.shape, device="cuda", generator=gen))]
    val = torch.randint(-3, 4, col.shape, device="cuda", generator=gen, dtype=torch.int8)
    return rp.to(torch.int32), col.to(torch.int32), val, gen


def _run(lens, n, ncols, dtype, sweep, pad=0, beta=0.5, ascending=True, nan=False):
    rp, col, val, gen = _matrix(lens, n, ncols + len(lens), ascending)
    val, m = val.to(dtype), rp.numel() - 1
    B = torch.randint(-3, 4, (n, ncols + pad), device="cuda", generator=gen, dtype=torch.int8).to(dtype)
    C = 2 * torch.randint(-3, 4, (m, ncols + 2 * pad), device="cuda", generator=gen, dtype=torch.int8).to(dtype)
    if nan:  # reaches the rows that hold its column, and no others
        B[n // 3], B[n // 2] = float("nan"), float("inf")
        val[val == 0] = 1
    if beta == 0.0:
        C.fill_(float("nan"))
    ref = C.clone()
    ends = rp.long()
    for c in range(ncols):
        b = B[:, c].double()
        if nan:
            b = torch.nan_to_num(b, nan=0.0, posinf=0.0)
        s = torch.cumsum(torch.cat([torch.zeros(1, device="cuda", dtype=torch.float64), val.double() * b[col.long()]]), 0)
        y = 2.0 * (s[ends[1:]] - s[ends[:-1]]).to(dtype)
        ref[:, c] = y if beta == 0.0 else y + beta * C[:, c]
    plan = capi.Plan(True, capi.SPMM_DEFAULT, dtype, m, n, col.numel(), rp, ncols=ncols, col=col, val=val)
    assert plan.info("sweep") == sweep, (m, n, ncols)
    capi.spmm(rp, col, val, B, C, ncols, 2.0, beta, plan=plan, ldb=ncols + pad, ldc=ncols + 2 * pad, k=n)
    plan.destroy()
    if nan:
        row = torch.repeat_interleave(torch.arange(m, device="cuda"), ends[1:] - ends[:-1])
        hit = torch.zeros(m, dtype=torch.bool, device="cuda")
        hit[row[(col == n // 3) | (col == n // 2)]] = True
        assert 0 < int(hit.sum()) < m // 10
        assert not torch.isfinite(C[hit][:, :ncols]).any()
        C, ref = C[~hit], ref[~hit]
    assert torch.equal(C[:, :ncols], ref[:, :ncols]), (m, n, ncols)
    if pad and beta != 0.0:
        assert torch.equal(C[:, ncols:], ref[:, ncols:])


def _rows(ncols, sv, per):
    """The smallest B the kernel takes with rows of `per`, not a round number."""
    b = ncols * sv
    return max(40003, 20_100_000 // b) if b % 128 == 0 else (9_100_000 if per >= 14 else 14_100_000) // b + 1


WIDTHS = [(torch.float32, n) for n in (17, 31, 32, 33, 47, 64, 65, 101, 128, 129, 255, 257, 300)] + [(torch.float64, n) for n in (9, 16, 17, 33, 65, 129)]


@pytest.mark.parametrize("dtype,ncols", WIDTHS)
def test_widths_of_b(dtype, ncols):
    sv = 4 if dtype == torch.float32 else 8
    n = _rows(ncols, sv, 17)
    _run([17] * (n // 5), n, ncols, dtype, 1, pad=3)
    rng = np.random.default_rng(ncols)
    _run(rng.integers(0, 2 * 16 + 9, n // 3), n, ncols, dtype, 1, beta=0.0)  # up to 40 with a mean of 20: what a wave stages differs


@pytest.mark.parametrize("dtype,ncols", [(torch.float32, 20), (torch.float32, 50), (torch.float32, 100), (torch.float64, 100)])
@pytest.mark.parametrize("per", [5, 16, 63])
@pytest.mark.parametrize("of_n", [0.5, 1.3, 3.1])
def test_rows_of_c_a_group_holds(dtype, ncols, per, of_n):
    n = _rows(ncols, 4 if dtype == torch.float32 else 8, per)
    _run([per] * int(n * of_n), n, ncols, dtype, 1)


def test_a_wave_that_stages_its_rows_in_several_turns():
    """Stretches of rows twice as long as the mean between stretches of empty ones."""
    lens = np.tile(np.r_[np.full(200, 40), np.zeros(200, int)], 150)
    _run(lens, 30011, 100, torch.float32, 1)
    _run(lens, 30011, 51, torch.float64, 1)


@pytest.mark.parametrize("dtype,ncols", [(torch.float32, 100), (torch.float64, 17)])
def test_nan_and_inf_stay_in_their_rows(dtype, ncols):
    n = _rows(ncols, 4 if dtype == torch.float32 else 8, 16)
    _run([16] * n, n, ncols, dtype, 1, nan=True)


def test_calls_that_stay_with_the_other_kernels():
    n = 30011
    _run([20] * n, n, 100, torch.float32, 0, ascending=False)
    _run([20] * (n - 1) + [49], n, 100, torch.float32, 0)  # a row longer than twice the mean and 8
    _run([3] * n, n, 150, torch.float32, 0)
    _run([20] * n, n, 64, torch.float32, 0)  # B of 7.7 MB
    _run([20] * 2000, n, 100, torch.float32, 0)  # too few rows to meet a row of B twice

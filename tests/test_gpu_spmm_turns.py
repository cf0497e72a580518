"""SpMM plans whose segments hold full turns of a wave's lane groups: rows of one length on both sides of what one group takes,
every number of lane groups, a matrix whose last segment is not full, rows too long for short segments (cut: usual segments
and the carry pass), and column and value arrays longer than the last row offset says.  Against float64 sums on the host;
tolerance: a row's products in another order, len u sum |a b| + 3 u |C|, u = 2^-24 or 2^-53."""
import numpy as np
import pytest
import torch

from library_amd import capi

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("per", [1, 7, 16, 17, 30, 32, 33, 64])
@pytest.mark.parametrize("case", ["even", "spare", "cut"])
def test_even_rows(dtype, per, case):
    rng = np.random.default_rng(per)
    m = (2_400_000 if case == "even" and per in (16, 17) else 300_000) // (per + 1) + 5
    reach, n = 3 * per + 40, m + 77
    lens = np.full(m, per)
    if case == "cut":
        lens[m // 3] = 1500
    rp = np.r_[0, np.cumsum(lens)].astype(np.int32)
    rows = np.repeat(np.arange(m), lens)
    col = np.minimum(rows + rng.integers(0, reach, rows.size), n - 1).astype(np.int32)
    col = col[np.lexsort((col, rows))]
    val = rng.uniform(-1, 1, col.size).astype(dtype)
    spare = 2001 if case == "spare" else 0
    d = [torch.from_numpy(a).cuda() for a in (rp, np.r_[col, np.zeros(spare, col.dtype)], np.r_[val, np.ones(spare, dtype)])]
    u = 2.0 ** (-53 if dtype == np.float64 else -24)
    for ncols in ((40, 64) if m > 100_000 else (1, 3, 8, 32, 64, 100)):
        B = rng.uniform(-1, 1, (n, ncols)).astype(dtype)
        C0 = rng.uniform(-1, 1, (m, ncols)).astype(dtype)
        plan = capi.Plan(True, capi.SPMM_DEFAULT, val.dtype, m, n, d[1].numel(), d[0], ncols=ncols, col=d[1], val=d[2])
        C = torch.from_numpy(C0.copy()).cuda()
        capi.spmm(*d, torch.from_numpy(B).cuda(), C, ncols, 1.5, 0.5, plan=plan, k=n)
        some = np.unique(np.r_[0, 1, m // 3, m - 1, rng.integers(0, m, 400)])
        got = C.cpu().numpy()
        for r in some:
            a, b = val[rp[r]:rp[r + 1]].astype(np.float64), B[col[rp[r]:rp[r + 1]]].astype(np.float64)
            size = 1.5 * (np.abs(a) @ np.abs(b)) + 0.5 * np.abs(C0[r])
            assert np.all(np.abs(got[r] - (1.5 * (a @ b) + 0.5 * C0[r])) <= (lens[r] + 6) * u * size + 1e-300), (ncols, r)
        if dtype == np.float32 and ncols == 64:  # every row, against a product in twice the precision
            ref = torch.from_numpy(C0).cuda().double() * 0.5
            ref.index_add_(0, torch.from_numpy(rows).cuda(), 1.5 * d[2][:col.size].double()[:, None] * torch.from_numpy(B).cuda().double()[d[1][:col.size].long()])
            assert (C.double() - ref).abs().max().item() <= (lens.max() + 6) * u * (1.5 * lens.max() + 0.5)
        plan.destroy()

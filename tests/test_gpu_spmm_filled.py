"""SpMM segments that are longer than usual because rows are long for the number of lane groups: calls without a plan and plans that have
not seen the columns, rows that segments cut among them.  Products of small integers, whose sums are exact in both types and in any order,
against integer sums."""
import numpy as np
import pytest
import torch

from library_amd import capi
from test_gpu_spmm_sweep import _matrix

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype,ncols,m,per,items", [
    (torch.float32, 256, 9001, 61, 512), (torch.float32, 128, 14001, 36, 256), (torch.float64, 96, 12001, 36, 256), (torch.float64, 64, 16001, 61, 256),
    (torch.float32, 128, 30001, 20, 128), (torch.float64, 27, 3144, 62, 128), (torch.float32, 21, 51556, 55, 256)])
@pytest.mark.parametrize("uneven", [False, True])
def test_rows_that_are_long_for_the_lane_groups(dtype, ncols, m, per, items, uneven):
    lens, n = np.full(m, per), 15001
    if uneven:  # some that cover several segments, some empty
        lens[::97], lens[5::101], lens[[3, m // 2]] = 0, 2 * per, 5000
    rp, col, val, gen = _matrix(lens, n, m)
    val, ends = val.to(dtype), rp.long()
    B = torch.randint(-3, 4, (n, ncols), device="cuda", generator=gen, dtype=torch.int8).to(dtype)
    C = 2 * torch.randint(-3, 4, (m, ncols), device="cuda", generator=gen, dtype=torch.int8).to(dtype)
    start, ref = C.clone(), C.clone()
    for c in range(ncols):
        s = torch.cumsum(torch.cat([torch.zeros(1, device="cuda", dtype=torch.float64), val.double() * B[:, c].double()[col.long()]]), 0)
        ref[:, c] = 2.0 * (s[ends[1:]] - s[ends[:-1]]).to(dtype) + 0.5 * C[:, c]
    capi.spmm(rp, col, val, B, C, ncols, 2.0, 0.5, k=n)
    assert torch.equal(C, ref)
    plan = capi.Plan(True, capi.SPMM_DEFAULT, dtype, m, n, col.numel(), rp, ncols=ncols)
    if not uneven:
        assert plan.info("segment_items") == items
    capi.spmm(rp, col, val, B, start, ncols, 2.0, 0.5, plan=plan, k=n)
    plan.destroy()
    assert torch.equal(start, ref)

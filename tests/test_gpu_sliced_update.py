"""New values for a sliced plan where a block of 4096 stored elements meets few of many slices, a run or hundreds of them: multiplies
with small integers, whose sums are exact, against integer sums."""
import numpy as np
import pytest
import torch

from library_amd import capi
from test_gpu_spmm_sweep import _matrix

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.float32, torch.float64])
@pytest.mark.parametrize("cols,per,reach", [
    (2200003, 5, 20000),   # 68 and 135 slices, one to four of them a block
    (4300007, 3, 300),     # 132 and 263, one or two
    (4300007, 3, 2000000),  # a third or a sixth of them, some by one element
    (9000011, 2, None)])   # 275 and 550, nearly all
def test_few_of_many_slices(dtype, cols, per, reach):
    m = cols // 4
    lens = np.full(m, per)
    lens[1000:90000] = 0
    lens[m // 2] = 9001 if reach is None or reach > 9001 else 500
    rp, col, val, gen = _matrix(lens, cols if reach is None else 2 * reach + 1, cols)
    ends = rp.long()
    if reach is not None:  # around the diagonal
        row = torch.repeat_interleave(torch.arange(m, device="cuda"), ends[1:] - ends[:-1])
        col = (col.long() + (row * 4 - reach).clamp(0, cols - 2 * reach - 1)).to(torch.int32)
    x = torch.randint(-3, 4, (cols,), device="cuda", generator=gen, dtype=torch.int8).to(dtype)
    y = torch.empty(m, dtype=dtype, device="cuda")
    plan = capi.Plan(False, capi.SPMV_SLICED, dtype, m, cols, col.numel(), rp, col=col, val=val.to(dtype))
    for turn in range(2):
        new = torch.randint(-3, 4, val.shape, device="cuda", generator=gen, dtype=torch.int8).to(dtype)
        plan.update_values(new)
        capi.spmv(rp, col, new, x, y, 1.0, 0.0, plan=plan)
        s = torch.cumsum(torch.cat([torch.zeros(1, device="cuda", dtype=torch.float64), new.double() * x.double()[col.long()]]), 0)
        assert torch.equal(y.double(), s[ends[1:]] - s[ends[:-1]]), turn
    plan.destroy()

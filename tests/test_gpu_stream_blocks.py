"""Row blocks of the stream kernel made along with the row-length histogram (plans that may look at the columns) against those
searched for one by one (plans that name the kernel): the same blocks give the same bits.  Sizes on and beside multiples of a
block, empty rows at either end and in long runs, column and value arrays longer than the last row offset says."""
import numpy as np
import pytest
import torch

from conftest import csr_from_lengths
from library_amd import capi

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape", ["multiple", "ragged", "spare", "gaps"])
def test_marked_blocks_equal_searched_ones(shape):
    rng = np.random.default_rng(5)
    lens = np.full(196608, 16)
    if shape == "ragged":
        lens = np.r_[np.zeros(5, int), rng.integers(8, 25, 200001), np.zeros(700, int)]
    elif shape == "gaps":
        lens[1000:4000] = 0
        lens[-1] = 3
    rp, col, val = csr_from_lengths(lens, 400000, 3, np.float64)
    if shape == "spare":
        col, val = np.r_[col, np.zeros(3001, col.dtype)], np.r_[val, np.ones(3001)]
    x, y0 = rng.uniform(-1, 1, 400000), rng.uniform(-1, 1, lens.size)
    d = [torch.from_numpy(a).cuda() for a in (rp, col, val, x)]
    out = []
    for alg in (capi.SPMV_DEFAULT, capi.SPMV_STREAM):
        plan = capi.Plan(False, alg, val.dtype, lens.size, x.size, col.size, d[0], col=d[1], val=d[2])
        assert plan.alg == capi.SPMV_STREAM
        y = torch.from_numpy(y0).cuda()
        capi.spmv(*d, y, 1.5, 0.5, plan=plan)
        out.append(y.cpu())
        plan.destroy()
    assert torch.equal(*out)

"""Transposes whose buckets of columns hold a little less and a little more than what 512 and 1024 threads sort in one turn, alone and
beside buckets of several turns and empty ones.  Integers and copied values: equal to a stable sort by column."""
import numpy as np
import pytest
import torch

from library_amd import capi

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.float32, torch.float64])
@pytest.mark.parametrize("n,nnz,turns", [
    (300000, 4000003, ()),               # buckets of 512 columns and about 6800 elements: 1024 threads
    (300000, 4000003, (8191, 8192, 8193, 20000, 0)),
    (1000003, 2000003, (4095, 4096, 4097, 9000, 0)),  # of about 2000: 512 threads
    (2000003, 1500001, ())])             # 2048 columns a bucket
def test_buckets_of_one_and_several_turns(dtype, n, nnz, turns):
    rng = np.random.default_rng(nnz)
    col = rng.integers(0, n, nnz).astype(np.int32)
    span = 512 if n < 1000000 else 1024
    for b, count in enumerate(turns):  # bucket 3 + 2 b holds `count` elements, wherever buckets of `span` columns start
        lo = (3 + 2 * b) * span
        col[(col >= lo) & (col < lo + span)] = n - 1 - b
        col[rng.choice(nnz, count, replace=False)] = lo + rng.integers(0, span, count)
    val, m = rng.uniform(-1, 1, nnz), nnz // 11
    rp = np.zeros(m + 1, np.int32)
    rp[1:-1], rp[-1] = np.sort(rng.integers(0, nnz + 1, m - 1)), nnz
    d = [torch.from_numpy(rp).cuda(), torch.from_numpy(col).cuda(), torch.from_numpy(val).cuda().to(dtype)]
    rows = torch.repeat_interleave(torch.arange(m, dtype=torch.int32), torch.from_numpy(np.diff(rp)).long()).cuda()
    got = capi.csr_transpose(*d, n)
    order = torch.sort(d[1], stable=True)[1]
    assert int(got[0][0]) == 0
    assert torch.equal(got[0][1:], torch.cumsum(torch.bincount(d[1], minlength=n), 0).to(torch.int32))
    assert torch.equal(got[1], rows[order])
    assert torch.equal(got[2], d[2][order])

"""Transposes whose buckets of columns hold a little less and a little more than what 512 and 1024 threads sort in one turn, alone and
beside buckets of several turns and empty ones, with every number of columns a bucket that has a kernel of its own.  Integers and copied
values: equal to a stable sort by column."""
import numpy as np
import pytest
import torch

from library_amd import capi

pytestmark = pytest.mark.gpu


def _shift(n, nnz):
    """Columns of a bucket, as a power of two (bucket_shift of asx_convert.hip)."""
    most, shift = min(7600.0, max(1024.0, nnz / 256.0)), 0
    while shift < 12 and nnz / -(-n // (2 << shift)) <= most:
        shift += 1
    while -(-n // (1 << shift)) > 1024:
        shift += 1
    return shift


@pytest.mark.parametrize("dtype", [torch.float32, torch.float64])
@pytest.mark.parametrize("n,nnz,shift,mean,turns", [
    (300000, 4000003, 9, 6825, ()),                                    # 1024 threads
    (300000, 4000003, 9, 6825, (8191, 8192, 8193, 20000, 0, 1)),
    (300000, 6000001, 9, 10238, ()),                                   # 1024 threads, several turns for most
    (300000, 6000001, 9, 10238, (8191, 8192, 8193, 4095, 4096, 4097)),
    (150000, 1000003, 9, 3412, (4095, 4096, 4097, 9000, 0, 1)),        # 512 threads and up to 512 columns
    (300000, 1000003, 10, 3412, (4095, 4096, 4097, 9000, 0, 1)),       # 1024
    (1000003, 2000003, 11, 4089, (4095, 4096, 4097, 9000, 0, 1)),      # 4096
    (2000003, 1500001, 12, 3067, (4095, 4096, 4097, 9000, 0, 1)),
    (2000003, 1500001, 12, 3067, ())])
def test_buckets_of_one_and_several_turns(dtype, n, nnz, shift, mean, turns):
    rng = np.random.default_rng(nnz)
    span, nbuckets = 1 << shift, -(-n >> shift)
    assert _shift(n, nnz) == shift and nnz // nbuckets == mean
    special = 3 + 2 * np.arange(len(turns))
    others = np.setdiff1d(np.arange(nbuckets - 1), special)
    col = others[rng.integers(0, len(others), nnz)] * span + rng.integers(0, span, nnz)
    chosen = np.split(rng.permutation(nnz)[:sum(turns)], np.cumsum(turns)[:-1]) if turns else []
    for b, at in zip(special, chosen):  # bucket b holds these elements and no others
        col[at] = b * span + rng.integers(0, span, len(at))
    assert tuple(np.bincount(col >> shift, minlength=nbuckets)[special]) == turns
    col = col.astype(np.int32)
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

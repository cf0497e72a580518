"""The transposed copy over the cases of its dispatch: few and many columns per bucket, buckets of one and of several
turns, a column that holds everything, more columns than the buckets take, one-based indices.  Integers and copied values:
bit-equal to numpy's stable sort by column."""
import numpy as np
import pytest
import torch

from library_amd import capi

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("m,n,nnz,shape", [
    (1, 1, 1, "even"), (5, 3, 4095, "even"), (300, 7, 4097, "even"), (1000, 1000, 60000, "even"), (20001, 511, 400003, "even"),
    (20000, 70001, 300000, "even"), (50000, 1200000, 500000, "even"), (3000, 4200001, 200000, "even"),
    (40000, 60000, 500000, "hub"), (70000, 1, 70000, "even"), (30000, 3000000, 400000, "hub"), (100, 50000, 90000, "last")])
def test_transpose_sizes(dtype, m, n, nnz, shape):
    rng = np.random.default_rng(nnz)
    rp = np.zeros(m + 1, np.int32)
    cuts = np.sort(rng.integers(0, nnz + 1, m - 1)) if m > 1 else np.empty(0, np.int64)
    rp[1:-1], rp[-1] = cuts, nnz
    col = rng.integers(0, n, nnz).astype(np.int32)
    if shape == "hub":
        col[rng.random(nnz) < 0.4] = n // 3
    elif shape == "last":
        col[:] = n - 1
    val = rng.uniform(-1, 1, nnz).astype(dtype)
    order = np.argsort(col, kind="stable")
    rows = np.repeat(np.arange(m, dtype=np.int32), np.diff(rp))
    rp_t = np.zeros(n + 1, np.int32)
    np.cumsum(np.bincount(col, minlength=n), out=rp_t[1:])
    for base in (0, 1):
        got = capi.csr_transpose(*[torch.from_numpy(a).cuda() for a in (rp + base, col + base, val)], n, idx_base=base)
        torch.cuda.synchronize()
        assert np.array_equal(got[0].cpu().numpy(), rp_t)
        assert np.array_equal(got[1].cpu().numpy(), rows[order])
        assert np.array_equal(got[2].cpu().numpy(), val[order])

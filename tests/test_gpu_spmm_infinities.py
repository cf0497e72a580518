"""The blocked SpMM kernel and infinities in B: a row of A whose 16 x 4 blocks hold every element meets no zero but its own,
so that an infinity it references arrives as that infinity - also in a block row's last block, where the kernel's batches
run past the end, and in B's last rows, where the last quad of rows is not full."""
import numpy as np
import pytest
import torch

from library_amd import capi

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("n", [7, 32, 64, 130])
@pytest.mark.parametrize("k", [4, 5, 6, 7, 8, 19, 36])
def test_infinity_in_a_full_block(dtype, n, k):
    m = 48
    rng = np.random.default_rng(k)
    val = rng.integers(1, 4, (m, k)).astype(dtype)
    B = rng.integers(-3, 4, (k, n)).astype(dtype)
    rp = np.arange(m + 1, dtype=np.int32) * k
    col = np.tile(np.arange(k, dtype=np.int32), m)
    d = [torch.from_numpy(a).cuda() for a in (rp, col, val.reshape(-1))]
    plan = capi.Plan(True, capi.SPMM_BLOCKED, val.dtype, m, k, col.size, d[0], ncols=n, col=d[1], val=d[2])
    for row in sorted({0, k // 2, (k - 1) // 4 * 4, k - 1}):
        Bi = B.copy()
        Bi[row, ::3] = np.inf
        C = torch.zeros(m * n, dtype=d[2].dtype, device="cuda")
        capi.spmm(*d, torch.from_numpy(Bi).cuda().reshape(-1), C, n, 1.0, 0.0, alg=capi.SPMM_BLOCKED, plan=plan, k=k)
        torch.cuda.synchronize()
        expect = val.astype(np.float64) @ B
        expect[:, ::3] = np.inf
        assert np.array_equal(C.cpu().numpy().reshape(m, n), expect), (k, row)
    plan.destroy()


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
def test_view_of_a_wider_matrix(dtype):
    """The kernel reads no row of B past the number that a call says or, where it does not, that the view of B tells."""
    m, n, k = 160, 40, 52
    rng = np.random.default_rng(3)
    val, B = (rng.integers(-3, 4, s).astype(dtype) for s in ((m, k), (k, 96)))
    d = [torch.from_numpy(a).cuda() for a in (np.arange(m + 1, dtype=np.int32) * k, np.tile(np.arange(k, dtype=np.int32), m), val.reshape(-1))]
    plan = capi.Plan(True, capi.SPMM_BLOCKED, d[2].dtype, m, k, m * k, d[0], ncols=n, col=d[1], val=d[2])
    view = torch.from_numpy(B).cuda()[:, 3:3 + n]
    for rows in (None, k):
        C = torch.zeros((m, n), dtype=d[2].dtype, device="cuda")
        capi.spmm(*d, view, C, n, 1.0, 0.0, alg=capi.SPMM_BLOCKED, plan=plan, ldb=96, k=rows)
        assert np.array_equal(C.cpu().numpy(), val @ B[:, 3:3 + n]), rows
    plan.destroy()

"""SpMM calls whose columns nobody has looked at: the device decides between the sweep kernel and the merge kernel, and rows that the
sweep leaves out are added by the merge kernel.  Products of small integers, whose sums are exact in both types and in any order,
against integer sums; what was decided is read from the call's workspace."""
import numpy as np
import pytest
import torch

from library_amd import capi
from test_gpu_spmm_sweep import _matrix

pytestmark = pytest.mark.gpu


def _answer(ws):
    """Where the answer lies in a workspace that was filled with 0x55, and what it says.  Behind it are four bytes that nobody writes, a
    byte for every workgroup of the sweep, 0 or 1, and what rounds the size up."""
    w = ws.cpu().numpy()
    i = int(np.flatnonzero(w != 0x55)[-1]) + 1
    i = int(np.flatnonzero(w[:i] > 1)[-1]) + 1
    assert (w[i - 4:i] == 0x55).all()
    return i - 8, int(w[i - 8:i - 4].view(np.int32)[0])


def _run(lens, n, ncols, dtype, taken, beta=0.5, pad=0, reach=None, room=True, ascending=True):
    rp, col, val, gen = _matrix(lens, n if reach is None else 2 * reach + 1, 5 + len(lens), ascending)
    m, nnz, ends = rp.numel() - 1, col.numel(), rp.long()
    if reach is not None:  # around the diagonal
        row = torch.repeat_interleave(torch.arange(m, device="cuda"), ends[1:] - ends[:-1])
        col = (col.long() + (row * n // m - reach).clamp(0, n - 2 * reach - 1)).to(torch.int32)
    val = val.to(dtype)
    B = torch.randint(-3, 4, (n, ncols + pad), device="cuda", generator=gen, dtype=torch.int8).to(dtype)
    C = 2 * torch.randint(-3, 4, (m, ncols + pad), device="cuda", generator=gen, dtype=torch.int8).to(dtype)
    if beta == 0.0:
        C.fill_(float("nan"))
    ref = C.clone()
    for c in range(ncols):
        s = torch.cumsum(torch.cat([torch.zeros(1, device="cuda", dtype=torch.float64), val.double() * B[:, c].double()[col.long()]]), 0)
        y = 2.0 * (s[ends[1:]] - s[ends[:-1]]).to(dtype)
        ref[:, c] = y if beta == 0.0 else y + beta * C[:, c]
    need = [capi.lib().asx_spmm_workspace_bytes(alg, capi.value_type(dtype), m, nnz, ncols) for alg in (capi.SPMM_DEFAULT, capi.SPMM_MERGE)]
    assert need[0] == need[1]  # a buffer for one does for the other
    ws = torch.full((need[0],), 0x55, dtype=torch.uint8, device="cuda")
    start = C.clone()
    capi.spmm(rp, col, val, B, C, ncols, 2.0, beta, workspace=ws, ldb=ncols + pad, ldc=ncols + pad, k=n)
    at, answer = _answer(ws)
    assert answer == taken
    if not room:  # a workspace without the answer's place, and nothing behind it is written
        ws.fill_(0x55)
        C.copy_(start)
        capi.spmm(rp, col, val, B, C, ncols, 2.0, beta, workspace=ws[:at], ldb=ncols + pad, ldc=ncols + pad, k=n)
        assert bool((ws[at:] == 0x55).all())
    assert torch.equal(C[:, :ncols], ref[:, :ncols]) and (not pad or beta == 0.0 or torch.equal(C[:, ncols:], ref[:, ncols:]))
    # a plan that has not seen the columns takes the same way
    plan = capi.Plan(True, capi.SPMM_DEFAULT, dtype, m, n, nnz, rp, ncols=ncols)
    capi.spmm(rp, col, val, B, start, ncols, 2.0, beta, plan=plan, ldb=ncols + pad, ldc=ncols + pad, k=n)
    plan.destroy()
    assert torch.equal(start[:, :ncols], ref[:, :ncols])


SHAPES = [(torch.float32, 100, 150001, 25), (torch.float32, 256, 100003, 36), (torch.float64, 50, 110003, 33), (torch.float32, 301, 50021, 29)]


def _even(m, per):
    return np.full(m, per)


@pytest.mark.parametrize("dtype,ncols,m,per", SHAPES)
@pytest.mark.parametrize("beta", [0.0, 0.5])
def test_uniform_columns_are_swept(dtype, ncols, m, per, beta):
    _run(_even(m, per), m, ncols, dtype, 1, beta, pad=3)


@pytest.mark.parametrize("dtype,ncols,m,per", SHAPES)
def test_rows_the_sweep_leaves_out(dtype, ncols, m, per):
    lens, most = _even(m, per), 2 * per + 8
    lens[[0, 7, 8, 9, 1000, m // 3, m - 2, m - 1]] = [most + 1, 300, most, 5000, most + 2, 30000, 700, 1300]
    lens[2000:2300] = 0
    lens[30000:30040] = 200
    sampled = np.arange(64) * 2 + 1
    assert lens[m * sampled // 128].max() == per
    _run(lens, m, ncols, dtype, 1, 0.5, pad=1)
    _run(lens, m, ncols, dtype, 1, 0.0)


@pytest.mark.parametrize("dtype,ncols,m,per", SHAPES)
def test_other_matrices_stay_with_the_merge_kernel(dtype, ncols, m, per):
    rng = np.random.default_rng(m)
    _run(_even(m, per), m, ncols, dtype, 0, reach=m // 20)
    _run(_even(m, per), m, ncols, dtype, 0, ascending=False)
    uneven = np.minimum((rng.pareto(1.3, m) * per * 0.24 + per * 0.24).astype(int), 20000)
    uneven[rng.integers(0, m, m // 50)] += max(0, per * m - int(uneven.sum())) // (m // 50) + 1
    _run(uneven, m, ncols, dtype, 0)
    _run(_even(m, per), m, ncols, dtype, 1, room=False)  # then without room for an answer

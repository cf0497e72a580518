"""Rows that the SpMM sweep kernel sums in two or four stretches: lengths around the limit and uneven ones, every number of lanes that
comes with several stretches, and that the error is no larger than the merge kernel's, which sums such rows in as many parts.  Products
of small integers are exact in both types and in any order."""
import numpy as np
import pytest
import torch

from library_amd import capi
from test_gpu_spmm_asked import _run as _run_asked
from test_gpu_spmm_sweep import _matrix, _rows, _run

pytestmark = pytest.mark.gpu

# lanes a row of B takes and stretches of a long row: 16 and 4, 32 and 2, 32 and 4, 64 and 4 (rows of B on lines that the merge
# kernel takes 256 bytes at a time)
SHAPES = [(torch.float32, 50, 0), (torch.float64, 24, 0), (torch.float32, 100, 0), (torch.float64, 41, 0), (torch.float32, 128, 140003), (torch.float32, 256, 140003)]


@pytest.mark.parametrize("dtype,ncols,n", SHAPES)
@pytest.mark.parametrize("beta", [0.0, 0.5])
def test_rows_of_several_stretches(dtype, ncols, n, beta):
    n = n or _rows(ncols, 4 if dtype == torch.float32 else 8, 24)
    rng = np.random.default_rng(ncols)
    lens = rng.integers(0, 49, n // 2)
    lens[:6] = [31, 32, 33, 34, 35, 48]
    _run(lens, n, ncols, dtype, 1, pad=3, beta=beta)
    _run([33] * (n // 3), n, ncols, dtype, 1, beta=beta)
    _run([64] * (n // 3 + 5), n, ncols, dtype, 1, beta=beta)


def test_rows_that_other_kernels_sum_in_more_parts():
    _run(np.tile([36, 65], 80001), 160002, 32, torch.float32, 0)   # eight groups share a row of more than 64
    _run(np.tile([36, 65], 60001), 120002, 100, torch.float32, 0)  # as a workgroup does in the chunk kernel
    _run(np.tile([36, 64], 60001), 120002, 100, torch.float32, 1)


@pytest.mark.parametrize("dtype,ncols,m,per", [(torch.float32, 100, 90001, 49), (torch.float32, 200, 60001, 40), (torch.float64, 30, 110003, 46)])
def test_calls_without_a_plan(dtype, ncols, m, per):
    lens = np.full(m, per)
    lens[[0, 7, 8, 1000, m // 3, m - 1]] = [2 * per + 9, 2 * per + 8, 32, 33, 7000, 1]
    _run_asked(lens, m, ncols, dtype, 1, 0.5, pad=1)
    _run_asked(np.full(m, per), m, ncols, dtype, 1, 0.0)


@pytest.mark.parametrize("ncols,m,per", [(50, 100001, 40), (50, 100001, 64), (100, 94796, 49), (100, 120001, 33), (128, 140003, 40)])
@pytest.mark.parametrize("planned", [True, False])
def test_error_is_the_merge_kernels(ncols, m, per, planned):
    """Five million sums and more, whose rms error is theirs to a tenth of a percent where the parts are as many; with one sum a row it was
    1.3 to 1.7 times as large."""
    rp, col, val, gen = _matrix([per] * m, m, per)
    val = torch.rand(val.shape, device="cuda", generator=gen) * 2 - 1
    B = torch.rand((m, ncols), device="cuda", generator=gen) * 2 - 1
    C = torch.empty((m, ncols), device="cuda")
    ref = torch.empty((m, ncols), dtype=torch.float64, device="cuda")
    for c in range(ncols):
        ref[:, c] = (val.double() * B[:, c].double()[col.long()]).view(m, per).sum(1)
    err = {}
    for alg in (capi.SPMM_MERGE, capi.SPMM_DEFAULT):
        plan = capi.Plan(True, alg, torch.float32, m, m, col.numel(), rp, ncols=ncols, col=col, val=val) if planned else None
        if planned and alg == capi.SPMM_DEFAULT:
            assert plan.info("sweep") == 1
        C.fill_(float("nan"))
        capi.spmm(rp, col, val, B, C, ncols, 1.0, 0.0, plan=plan, alg=alg)
        err[alg] = float((C.double() - ref).square().mean().sqrt())
        if plan:
            plan.destroy()
    assert err[capi.SPMM_DEFAULT] <= 1.05 * err[capi.SPMM_MERGE]

"""Where DEFAULT regroups scattered columns below four million stored elements: matrices whose slices hold many elements of a row
are faster in slices (60363 x 37: 14.1 us against 17.2 row-ordered), those whose slices hold few are not (61822 x 34 over three
times the columns: 18.0 against 16.6)."""
import pytest
import torch

from library_amd import capi

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows, cols, per_row, regrouped", [(60363, 37213, 37, True), (61822, 120316, 34, False)])
def test_default_regroups_scattered_columns(rows, cols, per_row, regrouped):
    gen = torch.Generator(device="cuda").manual_seed(1)
    rp = (torch.arange(rows + 1, device="cuda") * per_row).to(torch.int32)
    col = torch.randint(0, cols, (rows, per_row), device="cuda", generator=gen, dtype=torch.int32).sort(1)[0].reshape(-1).contiguous()
    val = torch.rand(rows * per_row, device="cuda", generator=gen, dtype=torch.float64)
    x, y = torch.rand(cols, device="cuda", generator=gen, dtype=torch.float64), torch.zeros(rows, device="cuda", dtype=torch.float64)
    plan = capi.Plan(False, capi.SPMV_DEFAULT, val.dtype, rows, cols, col.numel(), rp, col=col, val=val)
    assert (plan.alg == capi.SPMV_SLICED) == regrouped, plan.alg
    capi.spmv(rp, col, val, x, y, 1.0, 0.0, plan=plan)
    expect = (val * x[col.long()]).reshape(rows, per_row).sum(1)
    # positive products in another order: per_row u of the sum
    assert torch.all((y - expect).abs() <= 2 * per_row * 2.0**-53 * expect)
    plan.destroy()

"""Column-sliced plans at the limits of their sizes."""
import numpy as np
import pytest
import torch

from library_amd import capi

pytestmark = pytest.mark.gpu


def test_as_many_elements_as_slots_can_be_counted():
    """2^31 - 1 slots when the 255 that one slice may spare are counted.  Integers: exact in any order."""
    width, nnz = 32768, 2**31 - 1 - 255
    m = -(-nnz // width)
    row_ptr = torch.arange(m + 1, dtype=torch.int64, device="cuda") * width
    row_ptr[-1] = nnz
    row_ptr = row_ptr.to(torch.int32)
    col = torch.arange(width, dtype=torch.int32, device="cuda").repeat(m)[:nnz]
    val = torch.ones(nnz, dtype=torch.float32, device="cuda")
    x = (torch.arange(width, device="cuda") % 5).to(torch.float32)
    plan = capi.Plan(False, capi.SPMV_SLICED, val.dtype, m, width, nnz, row_ptr, col=col, val=val)
    y = torch.full((m,), -7.0, device="cuda")
    capi.spmv(row_ptr, col, val, x, y, 1.0, 0.0, plan=plan)
    torch.cuda.synchronize()
    plan.destroy()
    assert bool((y[:-1] == x.sum()).all()) and y[-1].item() == x[:nnz - (m - 1) * width].sum().item()
    with pytest.raises(capi.AsxError):
        capi.Plan(False, capi.SPMV_SLICED, val.dtype, m, width + 1, nnz, row_ptr, col=col, val=val)  # two slices
    capi.lib().asx_release_cached_memory()
    torch.cuda.empty_cache()


def test_steps_of_many_row_blocks_take_the_room_they_need():
    """100000 elements in 16 M rows and 1024 slices: tables of 67 MB by row block and slice, 5 MB for the rest, not 90 MB for
    the most steps that there could be."""
    m, n, nnz = 1 << 24, 1 << 25, 100000
    rng = np.random.default_rng(2)
    rows = np.sort(rng.choice(m, nnz, replace=False))
    row_ptr = torch.from_numpy(np.searchsorted(rows, np.arange(m + 1)).astype(np.int32)).cuda()
    col = torch.from_numpy(rng.integers(0, n, nnz).astype(np.int32)).cuda()
    val, x = torch.ones(nnz, device="cuda"), (torch.arange(n, device="cuda") % 5).to(torch.float32)
    y = torch.full((m,), -7.0, device="cuda")
    capi.lib().asx_release_cached_memory()
    before = torch.cuda.mem_get_info()[0]
    plan = capi.Plan(False, capi.SPMV_SLICED, val.dtype, m, n, nnz, row_ptr, col=col, val=val)
    capi.lib().asx_release_cached_memory()
    held = before - torch.cuda.mem_get_info()[0]
    capi.spmv(row_ptr, col, val, x, y, 1.0, 0.0, plan=plan)
    torch.cuda.synchronize()
    plan.destroy()
    expect = torch.zeros(m, device="cuda")
    expect[torch.from_numpy(rows).cuda()] = x[col.long()]
    assert torch.equal(y, expect)
    assert held < 110e6, held


@pytest.mark.parametrize("dtype", [torch.float32, torch.float64])
@pytest.mark.parametrize("m", [524289, 1048576, 1441793, 2097153, 2883585, 4194305, 5767169])
def test_row_blocks_of_every_size(m, dtype):
    """Matrices on which row blocks of 256 to 2048 rows begin, the last one of a single row.  Integers: exact in any order."""
    gen = torch.Generator(device="cuda").manual_seed(m)
    lens = torch.randint(0, 5, (m,), device="cuda", generator=gen)
    lens[-1], lens[m // 2] = 2, 70000
    row_ptr = torch.zeros(m + 1, dtype=torch.int32, device="cuda")
    row_ptr[1:] = torch.cumsum(lens, 0)
    nnz = int(row_ptr[-1])
    col = torch.randint(0, m, (nnz,), device="cuda", generator=gen, dtype=torch.int32)
    draw = lambda k: torch.randint(-3, 4, (k,), device="cuda", generator=gen).to(dtype)
    val, x, y = draw(nnz), draw(m), 2 * draw(m)
    rows = torch.repeat_interleave(torch.arange(m, device="cuda"), lens)
    ref = (2 * torch.zeros(m, dtype=torch.float64, device="cuda").index_add_(0, rows, (val * x[col.long()]).double()) + 0.5 * y).to(dtype)
    plan = capi.Plan(False, capi.SPMV_SLICED, dtype, m, m, nnz, row_ptr, col=col, val=val)
    capi.spmv(row_ptr, col, val, x, y, 2.0, 0.5, plan=plan)
    assert torch.equal(y, ref)
    if torch.cuda.get_device_properties(0).multi_processor_count == 256:
        sizes = {524289: (256, 256), 1048576: (256, 512), 1441793: (512, 1024), 2097153: (512, 1024), 2883585: (1024, 1024),
                 4194305: (1024, 2048), 5767169: (2048, 2048)}
        assert plan.info("rows_per_wave") == sizes[m][dtype == torch.float64]
    plan.destroy()

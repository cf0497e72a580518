"""As many stored elements as int32 offsets count: positions past the end of the last row do not fit int32."""
import pytest
import torch

from library_amd import capi

pytestmark = pytest.mark.gpu


def test_row_kernel():
    """Ones: 2048 a row, 2047 in the last, exact in float32."""
    nnz, m = 2**31 - 1, 1 << 20
    row_ptr = torch.arange(m + 1, dtype=torch.int64, device="cuda") * 2048
    row_ptr[-1] = nnz
    col = torch.zeros(nnz, dtype=torch.int32, device="cuda")
    val = torch.ones(nnz, dtype=torch.float32, device="cuda")
    C = torch.full((m, 1), -7.0, device="cuda")
    capi.spmm(row_ptr.to(torch.int32), col, val, torch.ones(1, device="cuda"), C, 1, 1.0, 0.0, alg=capi.SPMM_ROW)
    torch.cuda.synchronize()
    assert bool((C[:-1] == 2048.0).all()) and C[-1].item() == 2047.0

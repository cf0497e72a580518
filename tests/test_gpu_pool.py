"""Device memory that plans give back: destroying a plan while a stream is being captured, where that is allowed."""
import threading

import numpy as np
import pytest
import torch

from conftest import csr_from_lengths
from library_amd import capi

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("mode, other_thread", [("relaxed", False), ("relaxed", True), ("thread_local", True)])
def test_plan_destroyed_during_a_capture(mode, other_thread):
    """hipFree is allowed in these captures, so destroying a plan is: the capture survives and replays what it caught."""
    rp, col, val = csr_from_lengths(np.full(3000, 5), 4000, 1, np.float64)
    d = [torch.from_numpy(a).cuda() for a in (rp, col, val)]
    x, y = torch.rand(4000, dtype=torch.float64, device="cuda"), torch.zeros(3000, dtype=torch.float64, device="cuda")

    def plan():
        return capi.Plan(False, capi.SPMV_SLICED, val.dtype, 3000, 4000, col.size, d[0], col=d[1], val=d[2])
    kept, dropped = plan(), plan()
    workspace = torch.empty(max(kept.workspace_bytes, 256), dtype=torch.uint8, device="cuda")
    for p in (kept, dropped):
        capi.spmv(*d, x, y, 1.0, 0.0, plan=p, workspace=workspace)
    torch.cuda.synchronize()
    expect = y.clone()
    graph, side = torch.cuda.CUDAGraph(), torch.cuda.Stream()
    with torch.cuda.stream(side):
        with torch.cuda.graph(graph, stream=side, capture_error_mode=mode):
            capi.spmv(*d, x, y, 1.0, 0.0, plan=kept, workspace=workspace)
            if other_thread:
                t = threading.Thread(target=dropped.destroy)
                t.start()
                t.join()
            else:
                dropped.destroy()
            capi.spmv(*d, x, y, 1.0, 1.0, plan=kept, workspace=workspace)
    torch.cuda.synchronize()
    again = plan()  # over the memory that was given back
    for _ in range(3):
        y.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.allclose(y, 2 * expect, rtol=1e-15, atol=1e-15)
        capi.spmv(*d, x, y, 1.0, 0.0, plan=again, workspace=workspace)
        torch.cuda.synchronize()
        assert torch.equal(y, expect)
    del graph
    for p in (kept, again):
        p.destroy()

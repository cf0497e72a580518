"""The native calls from Python: what they get as a plan's handle (the address of a c_void_p, an adopted plan's integer, nothing
for a destroyed plan) and which errors wrong arguments raise."""
import ctypes as C

import pytest
import torch

from library_amd import capi


@pytest.mark.parametrize("h, address", [(None, None), (0x1230, 0x1230), (C.c_void_p(0x4560), 0x4560), (C.c_void_p(), None)])
def test_handle_of(h, address):
    assert capi._handle(h) == address


class _Tensor:
    """What the calls ask of a tensor; no address is followed, for every call below ends before the library is reached."""
    dtype, device = torch.float32, torch.device("cpu")

    def __init__(self, n):
        self.n = n

    def numel(self):
        return self.n

    def element_size(self):
        return 4

    def data_ptr(self):
        return 64


GOOD = dict(row_ptr=_Tensor(3), col=_Tensor(4), val=_Tensor(4), alpha=1.0, beta=0.0, workspace=_Tensor(1 << 20))
SPMV = dict(GOOD, x=_Tensor(5), y=_Tensor(2))
SPMM = dict(GOOD, B=_Tensor(10), Cm=_Tensor(4), ncols=2)


@pytest.mark.parametrize("name, wrong, error", [
    ("row_ptr", None, AttributeError), ("col", None, AttributeError), ("col", 3, AttributeError), ("x", None, AttributeError),
    ("y", 3, AttributeError), ("B", None, AttributeError), ("Cm", "c", AttributeError), ("alpha", "a", C.ArgumentError),
    ("beta", None, C.ArgumentError), ("alg", 1.5, C.ArgumentError), ("n", "n", C.ArgumentError), ("ldb", "l", C.ArgumentError),
    ("ldc", 2.0, C.ArgumentError), ("k", "k", C.ArgumentError), ("ncols", None, C.ArgumentError), ("ldb", 0, ZeroDivisionError),
    ("workspace", 3, AttributeError), ("row_ptr", _Tensor(1 << 40), OverflowError)])
def test_wrong_arguments_raise_their_own_errors(name, wrong, error):
    for call, good in ((capi.spmv, SPMV), (capi.spmm, SPMM)):
        if name in good or name == "alg" or (name == "n") == (call is capi.spmv) and name in ("n", "ldb", "ldc", "k"):
            with pytest.raises(error):
                call(**dict(good, **{name: wrong}))


def test_values_of_a_plan_that_are_no_tensor():
    plan = capi.Plan.adopt(0x1230)
    for call in (plan.update_values, plan.refresh_if_changed):
        with pytest.raises(AttributeError):
            call(3)


@pytest.mark.parametrize("B, ncols, ldb, rows", [
    (torch.empty(1000, 64)[:, :8], 8, 64, 1000), (torch.empty(1000, 64)[:, 56:], 8, 64, 1000), (torch.empty(3, 64)[:, :8], 8, 64, 3),
    (torch.empty(1000, 64), 8, 64, 1000), (torch.empty(64000), 8, 64, 1000), (torch.empty(64000 - 56), 8, 64, 1000),
    (torch.empty(1000, 8), 8, None, 1000), (torch.empty(8000), 8, None, 1000), (torch.empty(7), 8, 64, 0), (torch.empty(0, 8), 8, 64, 0)])
def test_rows_of_b_when_the_caller_does_not_say(B, ncols, ldb, rows):
    seen = []
    signature = C.CFUNCTYPE(C.c_int, C.c_void_p, C.c_int, C.c_int32, C.c_int32, C.c_int32, C.c_int32, C.c_float, C.c_void_p,
                            C.c_void_p, C.c_void_p, C.c_void_p, C.c_int64, C.c_float, C.c_void_p, C.c_int64, C.c_void_p, C.c_size_t, C.c_void_p)
    fn = signature(lambda plan, alg, m, k, *rest: seen.append(k) or 0)
    calls = capi._loaded()
    from library_amd import _calls
    _calls.streams_from(lambda: 0, lambda device: 0)
    try:
        for k in (None, 17):
            assert calls.spmm(C.cast(fn, C.c_void_p).value, False, None, 0, torch.zeros(2, dtype=torch.int32), torch.zeros(1, dtype=torch.int32),
                              torch.zeros(1), B, torch.zeros(8), ncols, 1.0, 0.0, ldb, None, k, None) == 0
    finally:
        capi._fast = None  # the next call asks torch for its streams again
    assert seen == [rows, 17]

"""What the native calls get as a plan's handle: the address of a c_void_p, an adopted plan's integer, nothing for a destroyed plan."""
import ctypes as C

import pytest

from library_amd import capi


@pytest.mark.parametrize("h, address", [(None, None), (0x1230, 0x1230), (C.c_void_p(0x4560), 0x4560), (C.c_void_p(), None)])
def test_handle_of(h, address):
    assert capi._handle(h) == address

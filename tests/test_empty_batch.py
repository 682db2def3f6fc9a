"""A batch of no problems (CPU test): nothing to do, so no device is asked for."""

import ctypes as C

from ccpi.reconstruction import _lib


def test_empty_batch_needs_no_device():
    L = _lib.lib()
    geoms = (_lib.CcpiGeometry * 1)()
    ptrs = (C.c_void_p * 1)()
    assert L.ccpi_pb_cgls_batched(geoms, 0, ptrs, ptrs, 3, None, 0, None) == 0

"""Fields in memory that the runtime knows: a pinned array and a device array as the caller's side of
smx_set_psi and smx_get_psi, at a size that an ordinary array takes through the pinned ring.  Against the
same calls with an ordinary array, bit for bit."""
import ctypes as C

import numpy as np
import pytest

from helpers import cfg_reference
from oracle import oracle as O
from smectic3d_amd import Solver
from smectic3d_amd._lib import check, lib

pytestmark = pytest.mark.gpu



@pytest.mark.parametrize("where", ["pinned", "device"])
def test_field_in_memory_the_runtime_knows(where):
    """The memory comes from the runtime that the library runs on (its symbols are found through the library)."""
    hip = lib()
    alloc, free = (hip.hipHostMalloc, hip.hipHostFree) if where == "pinned" else (hip.hipMalloc, hip.hipFree)
    shape = (96, 192, 256)  # 38 MB
    psi = O.ic_noise(*shape, 3, 0.3)
    with Solver(cfg_reference(*shape)) as s:
        s.set_psi(psi)
        want = s.get_psi()
        mem, size = C.c_void_p(), C.c_size_t(psi.nbytes)
        assert (alloc(C.byref(mem), size, C.c_uint(0)) if where == "pinned" else alloc(C.byref(mem), size)) == 0

        def copy(dst, src):  # hipMemcpyDefault
            assert hip.hipMemcpy(C.c_void_p(dst), C.c_void_p(src), size, C.c_int(4)) == 0

        try:
            ptr = C.cast(mem, C.POINTER(C.c_double))
            copy(mem.value, psi.ctypes.data)
            check(lib().smx_set_psi(s._h, ptr, shape[2]))
            assert np.array_equal(s.get_psi(), want)
            got = np.zeros(shape)
            copy(mem.value, got.ctypes.data)
            check(lib().smx_get_psi(s._h, ptr, shape[2]))
            copy(got.ctypes.data, mem.value)
            assert np.array_equal(got, want)
        finally:
            assert free(mem) == 0

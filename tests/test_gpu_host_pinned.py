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
    torch = pytest.importorskip("torch")
    shape = (96, 192, 256)  # 38 MB
    psi = O.ic_noise(*shape, 3, 0.3)
    with Solver(cfg_reference(*shape)) as s:
        s.set_psi(psi)
        want = s.get_psi()
        t = torch.empty(shape, dtype=torch.float64, pin_memory=True) if where == "pinned" else \
            torch.empty(shape, dtype=torch.float64, device="cuda:0")
        t.copy_(torch.from_numpy(psi))
        torch.cuda.synchronize()
        ptr = C.cast(C.c_void_p(t.data_ptr()), C.POINTER(C.c_double))
        check(lib().smx_set_psi(s._h, ptr, shape[2]))
        assert np.array_equal(s.get_psi(), want)
        t.zero_()
        torch.cuda.synchronize()
        check(lib().smx_get_psi(s._h, ptr, shape[2]))
        assert np.array_equal(t.cpu().numpy(), want)

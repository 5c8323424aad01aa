"""Which path a Neumann box steps on where both tiles fit: two launches, or four passes where x lines of 256
leave one block a CU in both FP64 kernels; and the same steps on either, to FP64 rounding (1e-13)."""
import numpy as np
import pytest

from helpers import cfg_reference, rel_l2
from smectic3d_amd import Solver
from smectic3d_amd import _abi as A

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape,prec,launches", [
    ((256, 256, 384), A.SMX_FP64, 4), ((256, 384, 192), A.SMX_FP64, 4), ((256, 384, 256), A.SMX_FP64, 4),
    ((256, 256, 384), A.SMX_FP32_MIXED, 2), ((256, 256, 256), A.SMX_FP64, 2), ((256, 128, 384), A.SMX_FP64, 2),
    ((192, 256, 384), A.SMX_FP64, 2), ((384, 128, 384), A.SMX_FP64, 2), ((256, 256, 512), A.SMX_FP64, 2)])
def test_path_of_the_step(shape, prec, launches):
    print(shape, prec, flush=True)
    cfg = cfg_reference(*shape, bc=A.SMX_BC_NEUMANN, eps=0.5, beta=0.3, dt=0.02, nl_model=A.SMX_NL_CUBIC, precision=prec)
    psi = np.resize(np.random.default_rng(4).uniform(-0.3, 0.3, 1000003), shape)
    with Solver(cfg) as s:
        s.set_psi(psi)
        assert len(s.profile_step(1)) == launches
        if launches == 2 or prec != A.SMX_FP64:
            return
        s.set_psi(psi)
        s.step(2)
        got = s.get_psi()
        s.set_schedule([(8, 0)] + s.schedule()[1:])
        s.set_psi(psi)
        s.step(2)
        assert rel_l2(s.get_psi(), got) < 1e-13

"""Changes of a state's form at every division of the y length, with a ragged last block of rows: two steps in
two launches, two in four passes (the state and the carry brought to the standard form, FP32 in FP32), two in
two launches again, against the oracle.  Tolerances are the steps' (FP64 1e-11, FP32-mixed 2e-5)."""
import pytest

from helpers import cfg_reference, rel_l2
from oracle import oracle as O
from smectic3d_amd import Solver
from smectic3d_amd import _abi as A

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("prec", [A.SMX_FP64, A.SMX_FP32_MIXED])
@pytest.mark.parametrize("bc", [A.SMX_BC_PERIODIC, A.SMX_BC_NEUMANN])
@pytest.mark.parametrize("nx,ny", [(16, 16), (16, 32), (16, 48), (16, 64), (16, 96), (24, 96), (16, 128), (16, 192),
                                   (16, 256), (16, 384)])
def test_every_division(nx, ny, bc, prec):
    shape = (nx, ny, 24)
    print(shape, bc, prec, flush=True)
    cfg = cfg_reference(*shape, bc=bc, eps=0.5, beta=0.3, dt=0.05, nl_model=A.SMX_NL_CUBIC, precision=prec)
    psi = O.ic_noise(*shape, 11, 0.3)
    orc = O.Oracle(cfg)
    orc.set_psi(psi)
    orc.step(6)
    with Solver(cfg) as s:
        default = s.schedule()
        s.set_psi(psi)
        assert len(s.profile_step(1)) == 2
        s.set_psi(psi)
        s.step(2)
        s.set_schedule([(default[0][0] // 2, 0)] + default[1:])
        s.step(2)
        s.set_schedule(default)
        s.step(2)
        assert rel_l2(s.get_psi(), orc.get_psi()) < (1e-11 if prec == A.SMX_FP64 else 2e-5)

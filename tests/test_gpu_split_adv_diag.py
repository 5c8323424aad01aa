"""The four-launch advected step's path and diagnostics: every shape of the division of the y length runs the
four kernels (a shape sent to the fifteen launches fails here), and L1, energy and d psi/dt of the stepped
split-form state match the oracle.

Tolerances are the plain two-launch step's: FP64 energy 1e-12, L1 1e-9 (rounding of 1e-16 over differences of
1e-3 and more), d psi/dt 1e-10; FP32-mixed 1e-5, 1e-3, 1e-3, all relative.
"""
import pytest

from helpers import cfg_reference, rel_l2
from oracle import oracle as O
from smectic3d_amd import Solver
from smectic3d_amd import _abi as A
from test_gpu_advect import structured_ic
from test_gpu_split_adv import SHAPES, SLOTS

pytestmark = pytest.mark.gpu

BOUNDS = {A.SMX_FP64: (1e-12, 1e-9, 1e-10), A.SMX_FP32_MIXED: (1e-5, 1e-3, 1e-3)}


@pytest.mark.parametrize("shape", SHAPES)
@pytest.mark.parametrize("prec", [A.SMX_FP64, A.SMX_FP32_MIXED])
def test_path_and_diagnostics_of_every_division(shape, prec):
    print("split advected diagnostics", shape, prec, flush=True)
    force = A.SMX_FORCE_MU if shape[0] % 32 else A.SMX_FORCE_SH
    cfg = cfg_reference(*shape, dt=2e-3, advect=1, force_form=force, precision=prec)
    psi = structured_ic(shape)
    orc = O.Oracle(cfg)
    orc.set_psi(psi)
    orc.step(5)
    energy, l1, rate = BOUNDS[prec]
    with Solver(cfg) as s:
        s.set_psi(psi)
        assert [k for k, _, _ in s.profile_step(1)] == SLOTS
        s.set_psi(psi)
        s.step(5)
        assert abs(s.energy() - orc.energy()) < energy * abs(orc.energy())
        assert abs(s.l1() - orc.l1()) < l1 * orc.l1()
        assert rel_l2(s.dtpsi(), orc.dtpsi()) < rate


@pytest.mark.parametrize("prec", [A.SMX_FP64, A.SMX_FP32_MIXED])
def test_long_x_lines_take_the_fifteen_launches(prec):
    """nx = 512: no Stokes tile of 512 threads."""
    with Solver(cfg_reference(512, 16, 16, dt=2e-3, advect=1, precision=prec)) as s:
        s.set_psi(structured_ic((512, 16, 16)))
        assert len(s.profile_step(1)) == 15

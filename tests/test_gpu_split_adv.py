"""The advected periodic step in four launches (smx_split_adv.h): every division of the y length against
the oracle, at the smallest and largest x and z lengths whose tiles exist with it, and the changes between
the split form of the state, which carries d_y psi too, and the standard one.

Tolerances are those of the fifteen launches: FP64 relative L2(psi) 1e-10, FP32-mixed 2e-5.
"""
import sys

import numpy as np
import pytest

from helpers import cfg_reference, rel_l2
from oracle import oracle as O
from smectic3d_amd import Solver
from smectic3d_amd import _abi as A
from test_gpu_advect import structured_ic

pytestmark = pytest.mark.gpu

MANY = [(8, 0), (16, 0), (16, 0), (16, 0)]  # any schedule but the default one takes the fifteen launches
TOL = {A.SMX_FP64: 1e-10, A.SMX_FP32_MIXED: 2e-5}
SLOTS = ["k_zsplit_force", "k_xsplit_stokes", "k_zsplit_advnl", "k_xsplit_adv"]


def say(*a):
    print(*a, flush=True)
    sys.stdout.flush()


SHAPES = [(16, 16, 16), (256, 16, 24), (24, 32, 384), (32, 48, 32), (16, 64, 256), (48, 96, 16), (192, 96, 24),
          (24, 128, 48), (256, 128, 16), (32, 192, 96), (16, 256, 128), (192, 256, 16), (24, 384, 32), (64, 384, 16)]


@pytest.mark.parametrize("shape", SHAPES)
@pytest.mark.parametrize("prec", [A.SMX_FP64, A.SMX_FP32_MIXED])
def test_every_division_of_y_matches_oracle(shape, prec):
    force = A.SMX_FORCE_MU if shape[0] % 32 else A.SMX_FORCE_SH
    say("split advected", shape, prec, force)
    pen = dict(w_mid=1.0, mid_plane=shape[2] // 2) if shape[1] % 64 == 0 else {}
    cfg = cfg_reference(*shape, dt=2e-3, advect=1, force_form=force, precision=prec, **pen)
    psi = structured_ic(shape)
    orc = O.Oracle(cfg)
    orc.set_psi(psi)
    orc.step(5)
    with Solver(cfg) as s:
        s.set_psi(psi)
        s.step(5)
        say("  ", [k for k, _, _ in s.profile_step(1)][:4])
        s.set_psi(psi)
        s.step(5)
        assert rel_l2(s.get_psi(), orc.get_psi()) < TOL[prec]
        s.set_schedule(MANY)
        s.set_psi(psi)
        s.step(5)
        assert rel_l2(s.get_psi(), orc.get_psi()) < TOL[prec]


@pytest.mark.parametrize("prec", [A.SMX_FP64, A.SMX_FP32_MIXED])
@pytest.mark.parametrize("shape", [(16, 32, 24), (48, 96, 32)])
def test_changes_of_form_keep_the_state(tmp_path, prec, shape):
    """Steps on either path in turn, diagnostics and a checkpoint in either form: the oracle's run, and
    a resumed run equal to the one that was saved."""
    cfg = cfg_reference(*shape, dt=2e-3, advect=1, force_form=A.SMX_FORCE_MU, precision=prec)
    psi = structured_ic(shape)
    orc = O.Oracle(cfg)
    orc.set_psi(psi)
    orc.step(9)
    with Solver(cfg) as s:
        default = s.schedule()
        s.set_psi(psi)
        s.step(3)
        assert [k for k, _, _ in s.profile_step(1)] == SLOTS
        s.set_psi(psi)
        s.step(3)
        a = s.get_psi()
        s.set_schedule(MANY)
        assert np.array_equal(s.get_psi(), a)
        s.step(3)
        s.save_checkpoint(tmp_path / "standard")
        s.set_schedule(default)
        s.step(2)
        s.dtpsi()  # leaves the carried arrays alone
        s.energy()
        s.save_checkpoint(tmp_path / "split")
        s.step(1)
        want = s.get_psi()
        assert rel_l2(want, orc.get_psi()) < TOL[prec]
    with Solver(cfg) as r:
        r.load_checkpoint(tmp_path / "split")
        r.step(1)
        assert np.array_equal(r.get_psi(), want)
        r.load_checkpoint(tmp_path / "standard")
        r.step(3)
        assert np.array_equal(r.get_psi(), want)

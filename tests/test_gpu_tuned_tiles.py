"""Where the autotuner's tiles run: the step of grids without the two-launch form, and the adjoint of the
others.  Tolerances are the four-pass kernels' (FP64 1e-11, FP32-mixed 2e-5 relative L2 against the oracle).
"""
import numpy as np
import pytest

from helpers import cfg_reference, rel_l2
from oracle import oracle as O
from smectic3d_amd import Solver
from smectic3d_amd import _abi as A

pytestmark = pytest.mark.gpu

PRECS = [A.SMX_FP64, A.SMX_FP32_MIXED]


def cfg(shape, prec, **kw):
    d = dict(eps=0.5, beta=0.3, dt=0.05, nl_model=A.SMX_NL_CUBIC, precision=prec)
    d.update(kw)
    return cfg_reference(*shape, **d)


def candidates(capfd, monkeypatch, s):
    """Number of candidates that an autotuner run of s times."""
    monkeypatch.setenv("SMX_TUNE_VERBOSE", "1")
    capfd.readouterr()
    s.autotune(2)
    return capfd.readouterr().err.count("smx_autotune")


@pytest.mark.parametrize("prec", PRECS)
def test_only_kernels_that_the_handle_can_launch_are_timed(capfd, monkeypatch, prec):
    shape = (32, 48, 96)
    for kw in (dict(bc=A.SMX_BC_NEUMANN), dict(advect=1, dt=2e-3), dict(w_mid=1.0, mid_plane=48, dt=2e-3)):
        with Solver(cfg(shape, prec, **kw)) as s:
            base = s.schedule()
            assert candidates(capfd, monkeypatch, s) == 0, kw
            assert s.schedule() == base
    with Solver(cfg(shape, prec)) as s:  # its adjoint has tiles
        assert candidates(capfd, monkeypatch, s) > 4
    with Solver(cfg((16, 512, 32), prec, bc=A.SMX_BC_NEUMANN)) as s:  # steps in four passes
        assert candidates(capfd, monkeypatch, s) > 4


@pytest.mark.parametrize("prec", PRECS)
def test_an_installed_default_keeps_the_adjoints_tiles(prec):
    """A tuned handle's reported schedule, installed again or in another handle: the same gradient bit for
    bit, so the same tiles (several grids, so that picks other than the default ones are among them)."""
    for shape in ((32, 32, 64), (64, 64, 64), (128, 64, 32), (64, 128, 128)):
        psi = O.ic_noise(*shape, 5, 0.3)
        with Solver(cfg(shape, prec)) as a, Solver(cfg(shape, prec)) as b:
            a.autotune(5)
            want = a.adjoint_grad(psi, 6, 3)
            a.set_schedule(a.schedule())
            b.set_schedule(a.schedule())
            for s in (a, b):
                got = s.adjoint_grad(psi, 6, 3)
                assert np.array_equal(got[1], want[1]) and got[0] == want[0] and got[2:] == want[2:], shape

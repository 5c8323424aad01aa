"""Where the autotuner's tiles run: the step of grids without the two-launch form, and the adjoint of the
others.  Tolerances are the four-pass kernels' (FP64 1e-11, FP32-mixed 2e-5 relative L2 against the oracle).
"""
import pytest

from helpers import cfg_reference
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

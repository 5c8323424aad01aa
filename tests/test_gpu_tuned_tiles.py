"""Where the autotuner's tiles run: the step of grids without the two-launch form, and the adjoint of the
others.  Tolerances are the four-pass kernels' (FP64 1e-11, FP32-mixed 2e-5 relative L2 against the oracle).
"""
import numpy as np
import pytest

from helpers import cfg_reference, rel_l2
from oracle import oracle as O
from smectic3d_amd import Solver
from smectic3d_amd import _abi as A
from test_gpu_advect import structured_ic

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


@pytest.mark.parametrize("prec", PRECS)
@pytest.mark.parametrize("kw", [dict(), dict(bc=A.SMX_BC_NEUMANN), dict(advect=1, dt=2e-3),
                                dict(w_mid=1.0, mid_plane=16, dt=2e-3)])
@pytest.mark.parametrize("shape", [(16, 512, 32), (48, 512, 32)])
def test_tuned_tiles_are_reported_and_stepped(shape, kw, prec):
    """Grids without the two-launch form: the tuner leaves the state alone and reports what it installs, a second
    handle takes the same tiles, and steps under them are those of the same schedule installed by hand, bit for
    bit, and the oracle's."""
    print(shape, kw, prec, flush=True)
    c = cfg(shape, prec, **kw)
    psi = structured_ic(shape) if c.advect else O.ic_noise(*shape, 31, 0.05)
    orc = O.Oracle(c)
    orc.set_psi(psi)
    orc.step(6)
    with Solver(c) as a, Solver(c) as b, Solver(c) as d:
        a.set_psi(psi)
        a.step(3)
        before = a.get_psi()
        chosen = a.autotune(5)
        print("  chosen", chosen, flush=True)
        assert a.schedule() == chosen and b.autotune(5) == chosen
        assert np.array_equal(a.get_psi(), before)
        a.step(3)
        tol = 2e-5 if prec == A.SMX_FP32_MIXED else 1e-10 if c.advect else 1e-11  # the steps' own tests'
        assert rel_l2(a.get_psi(), orc.get_psi()) < tol
        d.set_schedule(chosen)
        for s in (b, d):
            s.set_psi(psi)
            s.step(6)
            assert len(s.profile_step(1)) == (15 if c.advect else 4)
            s.set_psi(psi)
            s.step(6)
        assert np.array_equal(b.get_psi(), d.get_psi())


@pytest.mark.parametrize("prec", PRECS)
@pytest.mark.parametrize("shape", [(32, 32, 64), (64, 64, 64), (16, 512, 32)])
def test_gradient_under_tuned_tiles(shape, prec):
    """The adjoint's tuned tiles against its default ones, to the kernels' rounding (J and dJ/dpsi0 1e-12 in FP64, 1e-5
    in FP32-mixed; the parameters' derivatives, sums of either sign that cancel to 1e-3 or 1e-4 of their terms, 1e-9
    and 1e-3), and against the oracle's adjoint (FP64, 1e-9)."""
    psi = O.ic_noise(*shape, 5, 0.3)
    c = cfg(shape, prec)
    with Solver(c) as s:
        J0, g0, e0, q0 = s.adjoint_grad(psi, 6, 3)
    with Solver(c) as s:
        s.autotune(5)
        J, g, e, q = s.adjoint_grad(psi, 6, 3)
    tol = 1e-12 if prec == A.SMX_FP64 else 1e-5
    assert abs(J - J0) < tol * abs(J0) and rel_l2(g, g0) < tol
    par = 1e-9 if prec == A.SMX_FP64 else 1e-3
    assert abs(e - e0) < par * max(1, abs(e0)) and abs(q - q0) < par * max(1, abs(q0))
    if prec == A.SMX_FP64:
        Jo, go, eo, qo = O.adjoint_grad(c, psi, 6)
        assert abs(J - Jo) < 1e-12 * abs(Jo) and rel_l2(g, go) < 1e-9
        assert abs(e - eo) < 1e-9 * max(1, abs(eo)) and abs(q - qo) < 1e-9 * max(1, abs(qo))

"""The two-launch Neumann step (smx_split_neu.h): every division of the y length against the oracle, at
the smallest and largest x and z lengths whose tiles exist with it, and the changes between the split
form of the state and the standard one.

Tolerances are those of the four-pass kernels: FP64 relative L2(psi) 1e-11 after 5 steps, FP32-mixed 2e-5.
"""
import sys

import numpy as np
import pytest

from helpers import cfg_reference, rel_l2
from oracle import oracle as O
from smectic3d_amd import Batch, Solver
from smectic3d_amd import _abi as A

pytestmark = pytest.mark.gpu

SLOTS = ["k_nsplit_z", "k_nsplit_x"]


def say(*a):
    print(*a, flush=True)
    sys.stdout.flush()


def four_pass(default):
    """A schedule that is not the default one."""
    return [(default[0][0] // 2, 0)] + default[1:]


def cfg_neu(shape, prec, **kw):
    return cfg_reference(*shape, bc=A.SMX_BC_NEUMANN, eps=0.5, beta=0.3, dt=0.05, nl_model=A.SMX_NL_CUBIC,
                         precision=prec, **kw)


SHAPES = [(16, 16, 16), (512, 16, 24), (24, 32, 512), (32, 48, 32), (16, 64, 384), (48, 96, 16), (256, 96, 24),
          (24, 128, 48), (256, 128, 16), (32, 192, 96), (96, 192, 24), (16, 256, 192), (192, 256, 16), (24, 384, 64),
          (64, 384, 16), (16, 384, 128)]


@pytest.mark.parametrize("shape", SHAPES)
@pytest.mark.parametrize("prec", [A.SMX_FP64, A.SMX_FP32_MIXED])
def test_every_division_of_y_matches_oracle(shape, prec):
    say("split neumann", shape, prec)
    cfg = cfg_neu(shape, prec)
    psi = O.ic_noise(*shape, 23, 0.3)
    orc = O.Oracle(cfg)
    orc.set_psi(psi)
    orc.step(5)
    with Solver(cfg) as s:
        s.set_psi(psi)
        s.step(5)
        assert [k for k, _, _ in s.profile_step(1)] == SLOTS
        s.set_psi(psi)
        s.step(5)
        err = rel_l2(s.get_psi(), orc.get_psi())
        say("  err", err)
        assert err < (1e-11 if prec == A.SMX_FP64 else 2e-5)
        assert abs(s.energy() - orc.energy()) < (1e-12 if prec == A.SMX_FP64 else 1e-5) * abs(orc.energy())
        assert abs(s.l1() - orc.l1()) < (1e-9 if prec == A.SMX_FP64 else 1e-3) * orc.l1()
        assert rel_l2(s.dtpsi(), orc.dtpsi()) < (1e-10 if prec == A.SMX_FP64 else 1e-3)


@pytest.mark.parametrize("prec", [A.SMX_FP64, A.SMX_FP32_MIXED])
@pytest.mark.parametrize("shape", [(32, 48, 64), (48, 96, 32), (64, 64, 64)])
def test_changes_of_form_keep_the_state(tmp_path, prec, shape):
    """Steps on either path in turn, a field read in either form, an autotuner run and checkpoints of
    both forms in between: the oracle's run, and a resumed one equal to the one that was saved."""
    cfg = cfg_neu(shape, prec)
    psi = O.ic_noise(*shape, 61, 0.3)
    orc = O.Oracle(cfg)
    orc.set_psi(psi)
    orc.step(12)
    tol = 1e-11 if prec == A.SMX_FP64 else 2e-5
    with Solver(cfg) as s:
        default = s.schedule()
        s.set_psi(psi)
        s.step(3)
        a = s.get_psi()
        s.set_schedule(four_pass(default))
        assert np.array_equal(s.get_psi(), a)  # the state changes form when a step needs it
        s.step(3)
        assert len(s.profile_step(1)) == 4
        s.set_psi(psi)
        s.step(6)
        s.save_checkpoint(tmp_path / "standard")
        s.set_schedule(default)
        s.step(3)
        s.autotune(2)
        assert s.schedule() == default
        s.save_checkpoint(tmp_path / "split")
        s.step(3)
        want = s.get_psi()
        assert rel_l2(want, orc.get_psi()) < tol
    assert (tmp_path / "standard").read_bytes()[:8] == b"SMXCKPT1"
    with Solver(cfg) as r:
        r.load_checkpoint(tmp_path / "split")
        r.step(3)
        assert np.array_equal(r.get_psi(), want)
        r.load_checkpoint(tmp_path / "standard")
        r.step(6)
        assert np.array_equal(r.get_psi(), want)


def test_batch_and_surface_from_the_split_form():
    shape = (32, 48, 64)
    cfg = cfg_neu(shape, A.SMX_FP64)
    psi = O.ic_noise(*shape, 7, 0.3)
    with Batch([cfg, cfg]) as b:
        for s in b.boxes:
            s.set_psi(psi)
        b.run(7, graph_steps=3)
        got = [s.get_psi() for s in b.boxes]
    with Solver(cfg) as s:
        s.set_psi(psi)
        s.step(7)
        assert np.array_equal(got[0], s.get_psi()) and np.array_equal(got[1], got[0])
        orc = O.Oracle(cfg)
        orc.set_psi(s.get_psi())
        (gz, gv, _, _), gf = s.surftrack(0.1)
        assert rel_l2(s.get_psi(), got[0]) == 0.0
    (oz, ov, _, _), of = orc.surftrack(0.1)
    assert gf == of and np.array_equal(gz, oz)
    np.testing.assert_allclose(gv, ov, rtol=0, atol=1e-9 * np.abs(ov).max())

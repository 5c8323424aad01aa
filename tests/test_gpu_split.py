"""The two-launch periodic step (smx_split.h): every division of the y length against the oracle, at
the smallest and largest x and z lengths whose tiles exist with it, and the changes between the split
form of the state and the standard one.

Tolerances are those of the four-pass kernels: FP64 relative L2(psi) 1e-11 after 5 steps, FP32-mixed
2e-5; a state that changes form is rounded once more (FP64: a few 1e-16 a change).
"""
import sys

import numpy as np
import pytest

from helpers import cfg_reference, rel_l2
from oracle import oracle as O
from smectic3d_amd import Batch, Solver
from smectic3d_amd import _abi as A

pytestmark = pytest.mark.gpu

FOUR_PASS = [(16, 0), (16, 0), (8, 0), (16, 0)]  # any schedule but the default one


def say(*a):
    print(*a, flush=True)
    sys.stdout.flush()


SHAPES = [(16, 16, 16), (512, 16, 24), (24, 32, 512), (32, 48, 32), (16, 64, 384), (48, 96, 16), (384, 96, 24),
          (24, 128, 48), (512, 128, 16), (32, 192, 96), (96, 192, 24), (16, 256, 192), (192, 256, 16), (24, 384, 64),
          (64, 384, 16), (16, 384, 128)]


@pytest.mark.parametrize("shape", SHAPES)
@pytest.mark.parametrize("prec", [A.SMX_FP64, A.SMX_FP32_MIXED])
def test_every_division_of_y_matches_oracle(shape, prec):
    say("split", shape, prec)
    cfg = cfg_reference(*shape, eps=0.5, beta=0.3, dt=0.05, nl_model=A.SMX_NL_CUBIC, precision=prec)
    psi = O.ic_noise(*shape, 23, 0.3)
    orc = O.Oracle(cfg)
    orc.set_psi(psi)
    orc.step(5)
    with Solver(cfg) as s:
        s.set_psi(psi)
        s.step(5)
        assert [k for k, _, _ in s.profile_step(1)] == ["k_zsplit", "k_xsplit"]
        s.set_psi(psi)
        s.step(5)
        err = rel_l2(s.get_psi(), orc.get_psi())
        say("  err", err)
        assert err < (1e-11 if prec == A.SMX_FP64 else 2e-5)
        assert abs(s.energy() - orc.energy()) < (1e-12 if prec == A.SMX_FP64 else 1e-5) * abs(orc.energy())
        assert abs(s.l1() - orc.l1()) < (1e-9 if prec == A.SMX_FP64 else 1e-3) * orc.l1()
        assert rel_l2(s.dtpsi(), orc.dtpsi()) < (1e-10 if prec == A.SMX_FP64 else 1e-3)


@pytest.mark.parametrize("prec", [A.SMX_FP64, A.SMX_FP32_MIXED])
def test_penalty_plane_and_quintic(prec):
    shape = (32, 48, 96)
    cfg = cfg_reference(*shape, dt=2e-3, w_mid=1.0, mid_plane=48, precision=prec)
    psi = O.ic_noise(*shape, 5, 0.3)
    orc = O.Oracle(cfg)
    orc.set_psi(psi)
    orc.step(10)
    with Solver(cfg) as s:
        s.set_psi(psi)
        s.step(10)
        assert rel_l2(s.get_psi(), orc.get_psi()) < (1e-11 if prec == A.SMX_FP64 else 2e-5)


@pytest.mark.parametrize("prec", [A.SMX_FP64, A.SMX_FP32_MIXED])
@pytest.mark.parametrize("shape", [(32, 48, 64), (48, 96, 32), (64, 64, 64)])
def test_changes_of_form_keep_the_state(prec, shape):
    """Steps on either path in turn, a field read in either form, an autotuner run in between: the
    oracle's run."""
    cfg = cfg_reference(*shape, eps=0.5, beta=0.3, dt=0.05, nl_model=A.SMX_NL_CUBIC, precision=prec)
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
        s.set_schedule(FOUR_PASS)
        assert np.array_equal(s.get_psi(), a)  # the state changes form when a step needs it
        s.step(3)
        s.set_schedule(default)
        s.step(3)
        s.autotune(2)
        assert s.schedule() == default
        s.step(3)
        assert rel_l2(s.get_psi(), orc.get_psi()) < tol


@pytest.mark.parametrize("prec", [A.SMX_FP64, A.SMX_FP32_MIXED])
def test_checkpoints_of_both_forms(tmp_path, prec):
    """A split-form file continues bit for bit; a standard-form one loads into a handle that steps in
    two launches."""
    shape = (32, 48, 64)
    cfg = cfg_reference(*shape, eps=0.5, beta=0.3, dt=0.05, nl_model=A.SMX_NL_CUBIC, precision=prec)
    psi = O.ic_noise(*shape, 62, 0.3)
    orc = O.Oracle(cfg)
    orc.set_psi(psi)
    orc.step(10)
    with Solver(cfg) as s:
        s.set_psi(psi)
        s.step(10)
        want = s.get_psi()
        s.set_psi(psi)
        s.step(4)
        s.save_checkpoint(tmp_path / "split")
        s.set_psi(psi)
        s.set_schedule(FOUR_PASS)
        s.step(4)
        s.save_checkpoint(tmp_path / "standard")
    assert (tmp_path / "standard").read_bytes()[:8] == b"SMXCKPT1"
    with Solver(cfg) as r:
        r.load_checkpoint(tmp_path / "split")
        r.step(6)
        assert np.array_equal(r.get_psi(), want)
        r.load_checkpoint(tmp_path / "standard")
        r.step(6)
        assert rel_l2(r.get_psi(), orc.get_psi()) < (1e-11 if prec == A.SMX_FP64 else 2e-5)


def test_batch_graph_spans_its_stretches():
    """A graph of up to four stretches; odd numbers of them and a remainder give the same steps."""
    cfgs = [cfg_reference(32, 48, 32, eps=0.5 + 0.01 * i, beta=0.3, dt=0.05, nl_model=A.SMX_NL_CUBIC) for i in range(3)]
    psis = [O.ic_noise(32, 48, 32, 70 + i, 0.3) for i in range(3)]
    with Batch(cfgs) as b:
        for s, p in zip(b.boxes, psis):
            s.set_psi(p)
        for n in (8, 5, 23, 2):  # 4 stretches of 2; 2 and a step; 11 and a step; 1
            b.run(n, graph_steps=2)
        got = [s.get_psi() for s in b.boxes]
    for c, p, g in zip(cfgs, psis, got):
        with Solver(c) as s:
            s.set_psi(p)
            s.step(38)
            assert rel_l2(g, s.get_psi()) < 1e-13

"""surfTrack from a state of the two-launch step: psi, the crossings and the z derivative come from the split
form itself where a z tile is whole waves, through the standard form elsewhere.  At every division of the y
length and at z lengths of either kind, against the oracle on the field that the handle returns, with the
tolerances of the standard-form path (FP64: crossings equal, values 1e-9 of the largest; FP32-mixed: the state's
own accuracy, 1e-6 of the largest, against the same call on a state set from that field)."""
import numpy as np
import pytest

from helpers import cfg_reference
from oracle import oracle as O
from smectic3d_amd import Solver
from smectic3d_amd import _abi as A

pytestmark = pytest.mark.gpu

SHAPES = [(16, 16, 64), (16, 32, 24), (24, 32, 192), (16, 48, 128), (16, 64, 48), (32, 64, 256), (16, 96, 96),
          (24, 96, 32), (16, 128, 64), (16, 192, 96), (24, 256, 64), (16, 384, 32), (16, 128, 384), (16, 64, 512)]


@pytest.mark.parametrize("bc", [A.SMX_BC_PERIODIC, A.SMX_BC_NEUMANN])
@pytest.mark.parametrize("shape", SHAPES)
def test_surftrack_of_a_stepped_state(shape, bc):
    print(shape, bc, flush=True)
    cfg = cfg_reference(*shape, bc=bc, eps=0.5, beta=0.3, dt=0.05, nl_model=A.SMX_NL_CUBIC)
    psi = O.ic_noise(*shape, 7, 0.4)
    orc = O.Oracle(cfg)
    orc.set_psi(psi)
    orc.step(3)
    (oz, ov, oh, ok), of = orc.surftrack(0.05)
    assert of > shape[0] * shape[1] // 4
    with Solver(cfg) as s:
        s.set_psi(psi)
        assert len(s.profile_step(1)) == 2
        s.set_psi(psi)
        s.step(3)
        before = s.get_psi()
        (gz, gv, gh, gk), gf = s.surftrack(0.05)
        assert np.array_equal(s.get_psi(), before)
        assert gf == of and np.array_equal(gz, oz)
        np.testing.assert_allclose(gv, ov, rtol=0, atol=1e-9 * np.abs(ov).max())
        # the curvatures divide by the gradient: relative to each value and to the middle of them
        for g, o in ((gh, oh), (gk, ok)):
            np.testing.assert_allclose(g, o, rtol=1e-6, atol=1e-9 * np.median(np.abs(o)))


@pytest.mark.parametrize("bc", [A.SMX_BC_PERIODIC, A.SMX_BC_NEUMANN])
@pytest.mark.parametrize("shape", SHAPES)
def test_mixed_state_matches_its_own_field(shape, bc):
    print(shape, bc, flush=True)
    cfg = cfg_reference(*shape, bc=bc, eps=0.5, beta=0.3, dt=0.05, nl_model=A.SMX_NL_CUBIC, precision=A.SMX_FP32_MIXED)
    c64 = cfg_reference(*shape, bc=bc, eps=0.5, beta=0.3, dt=0.05, nl_model=A.SMX_NL_CUBIC)
    with Solver(cfg) as s, Solver(c64) as r:
        s.set_psi(O.ic_noise(*shape, 7, 0.4))
        s.step(3)
        r.set_psi(s.get_psi())
        (gz, gv, _, _), gf = s.surftrack(0.05)
        (rz, rv, _, _), rf = r.surftrack(0.05)
        assert gf == rf and np.array_equal(gz, rz)
        np.testing.assert_allclose(gv, rv, rtol=0, atol=1e-6 * np.abs(rv).max())

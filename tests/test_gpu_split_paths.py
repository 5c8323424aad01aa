"""Which path a periodic box steps on where its tiles fit: two launches, or four passes in FP64 boxes of long x lines
with hardly any block in the x kernel."""
import pytest

from helpers import cfg_reference
from oracle import oracle as O
from smectic3d_amd import Solver
from smectic3d_amd import _abi as A

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape,prec,launches", [((512, 16, 16), A.SMX_FP64, 4), ((384, 16, 16), A.SMX_FP64, 4),
                                                 ((512, 16, 24), A.SMX_FP64, 2), ((384, 16, 24), A.SMX_FP64, 2),
                                                 ((256, 16, 16), A.SMX_FP64, 2), ((512, 16, 16), A.SMX_FP32_MIXED, 2)])
def test_path_of_long_lines_and_few_blocks(shape, prec, launches):
    cfg = cfg_reference(*shape, eps=0.5, beta=0.3, dt=0.05, nl_model=A.SMX_NL_CUBIC, precision=prec)
    with Solver(cfg) as s:
        s.set_psi(O.ic_noise(*shape, 5, 0.3))
        assert len(s.profile_step(1)) == launches

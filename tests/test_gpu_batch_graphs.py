"""The captured graphs of a batch: which calls capture, and that every mix of them makes the steps asked for.

Results against single boxes run step by step: 1e-13 relative in FP64, the grouped kernels' rounding.
"""
import pytest

from helpers import cfg_reference, rel_l2
from oracle import oracle as O
from smectic3d_amd import Batch, Solver
from smectic3d_amd import _abi as A

pytestmark = pytest.mark.gpu

SHAPE = (32, 48, 32)


def boxes(n=3):
    cfgs = [cfg_reference(*SHAPE, eps=0.5 + 0.01 * i, beta=0.3, dt=0.05, nl_model=A.SMX_NL_CUBIC) for i in range(n)]
    return cfgs, [O.ic_noise(*SHAPE, 70 + i, 0.3) for i in range(n)]


def check(cfgs, psis, got, steps):
    for c, p, g in zip(cfgs, psis, got):
        with Solver(c) as s:
            s.set_psi(p)
            s.step(steps)
            assert rel_l2(g, s.get_psi()) < 1e-13


@pytest.mark.parametrize("calls,nodes", [((8, 6, 8, 6, 2, 10), 16),  # four stretches, then three, one and five
                                         ((6, 8, 6), 12),            # three, then four
                                         ((2, 8, 2), None)])         # one, then four: the longer graph is added
def test_calls_of_other_lengths_capture_nothing_again(calls, nodes):
    """Two launches a step of a group, stretches of two steps: the longer graph stays as it was captured."""
    cfgs, psis = boxes()
    with Batch(cfgs) as b:
        for s, p in zip(b.boxes, psis):
            s.set_psi(p)
        seen = []
        for n in calls:
            b.run(n, graph_steps=2)
            seen.append(b.graph_nodes())
        print("nodes", seen, flush=True)
        if nodes is None:
            assert seen == [4, 16, 16]
        else:
            assert seen == [nodes] * len(calls)
        got = [s.get_psi() for s in b.boxes]
    check(cfgs, psis, got, sum(calls))


def test_another_stretch_captures_again():
    cfgs, psis = boxes()
    with Batch(cfgs) as b:
        for s, p in zip(b.boxes, psis):
            s.set_psi(p)
        b.run(8, graph_steps=2)
        b.run(5, graph_steps=5)
        assert b.graph_nodes() == 10
        b.run(9, graph_steps=3)
        assert b.graph_nodes() == 18
        got = [s.get_psi() for s in b.boxes]
    check(cfgs, psis, got, 22)


@pytest.mark.parametrize("prec", [A.SMX_FP64, A.SMX_FP32_MIXED])
def test_tiles_of_the_four_passes_do_not_divide_a_group(prec):
    """Boxes that step in two launches share them whatever their adjoint's tiles are: one box tuned, the
    group and its graph stay (two launches a step in all, four grids to have tiles other than the default)."""
    for shape in ((32, 32, 32), (64, 64, 64), (64, 96, 48), (96, 128, 64)):
        cfgs = [cfg_reference(*shape, eps=0.5, beta=0.3, dt=0.05, nl_model=A.SMX_NL_CUBIC, precision=prec)] * 3
        psi = O.ic_noise(*shape, 5, 0.3)
        with Batch(cfgs) as b:
            for s in b.boxes:
                s.set_psi(psi)
            b.boxes[0].autotune(3)
            b.run(4, graph_steps=4)
            print(shape, "nodes", b.graph_nodes(), flush=True)
            assert b.graph_nodes() == 2 * 4
            b.boxes[1].autotune(3)
            b.run(4, graph_steps=4)
            assert b.graph_nodes() == 2 * 4
            # boxes stepped in one group from equal states stay equal
            assert rel_l2(b.boxes[0].get_psi(), b.boxes[2].get_psi()) == 0.0

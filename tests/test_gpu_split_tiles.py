"""Tiles of the two-launch z kernels by their rows' padding and by the number of blocks: whole pieces of a y line in
FP32 from 192 blocks on (nx = 48 with 16 y2) and half pieces below, unpadded rows (12 values of a y line; 8 at
nz = 512), one column of padding (24 values), and the largest tile (24 values, nz = 384).  Against the oracle,
with the steps' tolerances (plain FP64 1e-11, advected 1e-10, FP32-mixed 2e-5); a group against single boxes to the
grouped kernels' rounding (2e-6)."""
import numpy as np
import pytest

from helpers import cfg_reference, rel_l2
from oracle import oracle as O
from smectic3d_amd import Batch, Solver
from smectic3d_amd import _abi as A
from test_gpu_advect import structured_ic

pytestmark = pytest.mark.gpu

WHOLE = [(nx, ny, nz) for ny, nz in ((192, 384), (192, 512), (384, 192), (384, 256)) for nx in (32, 48)]
PADS = [(16, 192, 256), (24, 192, 48), (16, 384, 128), (16, 384, 96), (16, 64, 512), (24, 96, 512), (16, 384, 384)]


def run(shape, prec, **kw):
    cfg = cfg_reference(*shape, eps=0.5, beta=0.3, nl_model=A.SMX_NL_CUBIC, precision=prec, **kw)
    psi = structured_ic(shape) if cfg.advect else O.ic_noise(*shape, 23, 0.3)
    orc = O.Oracle(cfg)
    orc.set_psi(psi)
    orc.step(3)
    with Solver(cfg) as s:
        s.set_psi(psi)
        assert len(s.profile_step(1)) == (4 if cfg.advect else 2)
        s.set_psi(psi)
        s.step(3)
        tol = 2e-5 if prec == A.SMX_FP32_MIXED else 1e-10 if cfg.advect else 1e-11
        assert rel_l2(s.get_psi(), orc.get_psi()) < tol
        assert abs(s.energy() - orc.energy()) < (1e-12 if prec == A.SMX_FP64 else 1e-5) * abs(orc.energy())
        if not cfg.advect:  # psi and the scan in one kernel
            (gz, _, _, _), gf = s.surftrack(0.05)
            (oz, _, _, _), of = orc.surftrack(0.05)
            if prec == A.SMX_FP64:
                assert gf == of and np.array_equal(gz, oz)


@pytest.mark.parametrize("kw", [dict(dt=0.05), dict(dt=2e-3, advect=1)])
@pytest.mark.parametrize("shape", WHOLE)
def test_whole_and_half_pieces(shape, kw):
    print(shape, kw, flush=True)
    run(shape, A.SMX_FP32_MIXED, **kw)


@pytest.mark.parametrize("prec", [A.SMX_FP64, A.SMX_FP32_MIXED])
@pytest.mark.parametrize("kw", [dict(dt=0.05), dict(dt=2e-3, advect=1)])
@pytest.mark.parametrize("shape", PADS)
def test_padding_of_a_tiles_rows(shape, kw, prec):
    print(shape, kw, prec, flush=True)
    run(shape, prec, **kw)


@pytest.mark.parametrize("shape,prec", [((256, 256, 16), A.SMX_FP64), ((384, 32, 16), A.SMX_FP64),
                                        ((384, 96, 24), A.SMX_FP64), ((384, 64, 16), A.SMX_FP32_MIXED),
                                        ((384, 64, 128), A.SMX_FP32_MIXED)])
def test_advected_x_kernels_of_long_lines(shape, prec):
    """FP64 Stokes on lines of 256 with 16 y2 and of 384; the FP32 update on lines of 384 with 36 and 260 blocks."""
    print(shape, prec, flush=True)
    run(shape, prec, dt=2e-3, advect=1)


def test_a_group_takes_the_tile_of_its_boxes():
    shape = (48, 192, 384)
    cfgs = [cfg_reference(*shape, eps=0.5 + 0.1 * i, beta=0.3, dt=0.05, nl_model=A.SMX_NL_CUBIC,
                          precision=A.SMX_FP32_MIXED) for i in range(2)]
    psis = [O.ic_noise(*shape, 70 + i, 0.3) for i in range(2)]
    with Batch(cfgs) as b:
        for s, p in zip(b.boxes, psis):
            s.set_psi(p)
        b.run(4, graph_steps=2)
        got = [s.get_psi() for s in b.boxes]
    for c, p, g in zip(cfgs, psis, got):
        with Solver(c) as s:
            s.set_psi(p)
            s.step(4)
            assert rel_l2(g, s.get_psi()) < 2e-6

"""Whole fields between host and device through the pinned ring: sizes below, at and above one chunk,
one and several workers in either direction, ragged last chunks, padded rows, and transfers from several threads at once.
Fields come back bit for bit (FP64) after a round trip through a state's transform pair to 1e-13."""
import threading

import numpy as np
import pytest

from helpers import cfg_reference, rel_l2
from oracle import oracle as O
from smectic3d_amd import Solver

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape", [(32, 32, 48), (64, 32, 64), (64, 64, 64), (96, 96, 128), (192, 96, 384)])
def test_round_trip(shape):
    psi = O.ic_noise(*shape, 3, 0.3)
    with Solver(cfg_reference(*shape)) as s:
        s.set_psi(psi)
        a = s.get_psi()
        assert rel_l2(a, psi) < 1e-13
        assert np.array_equal(s.get_psi(), a)  # another destination, the same values
        nz = shape[2]
        b = s.get_psi(row_stride=nz + 2).reshape(-1, nz + 2)[:, :nz].reshape(shape)
        assert np.array_equal(b, a)


def test_transfers_from_several_threads():
    shape = (128, 128, 256)
    psis = [O.ic_noise(*shape, 20 + i, 0.3) for i in range(4)]
    errs = [None] * 4

    def run(i):
        with Solver(cfg_reference(*shape)) as s:
            worst = 0.0
            for _ in range(5):
                s.set_psi(psis[i])
                worst = max(worst, rel_l2(s.get_psi(), psis[i]))
            errs[i] = worst

    threads = [threading.Thread(target=run, args=(i,)) for i in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert all(e is not None and e < 1e-13 for e in errs), errs

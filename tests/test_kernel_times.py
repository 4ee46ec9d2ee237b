"""Asking for kernel times leaves a 1D step the launches it has without."""
from __future__ import annotations

import numpy as np
import pytest

from gamma_amd import hip, setups as S


@pytest.mark.gpu
@pytest.mark.parametrize("mk", [lambda: S.shock_tube_1d(200), lambda: S.blandford_mckee_1d(300)])
def test_gpu_1d_timed_steps_are_the_ordinary_ones(mk):
    g, plain = hip.Grid(mk()), hip.Grid(mk())
    g.kernel_times()
    for k in (3, 50):                      # the second past the events kept before they are read back
        g.step(k)
        plain.step(k)
        ms, n = g.kernel_times()
        assert n[1] == k and n[0] == 3 * k and not n[2:].any()
        assert 0. < ms[0] < 10. and 0. < ms[1] < 10.
    for f in (S.RHO, S.PPP, S.UU1, hip.F_X):
        assert np.array_equal(g.cells(f), plain.cells(f), equal_nan=True), f

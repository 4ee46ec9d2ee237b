"""Grids of few long tracks, whose passes over a track run on the whole chip:
bit for bit the oracle's run, with splits and merges."""
from __future__ import annotations

import dataclasses

import numpy as np
import pytest

from gamma_amd import hip, setups as S
import oracle_ctypes as oc


def _equal(s, steps):
    g, o = hip.Grid(s), oc.OracleGrid(s)
    for k in steps:
        g.step(k)
        o.run(k)
        for f in (S.RHO, S.PPP, S.UU1, hip.F_X, hip.F_DX):
            a, b = np.concatenate(g.active(f)), np.concatenate(o.active(f))
            assert np.array_equal(a, b, equal_nan=True), (f, k)
        assert np.array_equal(g.tracks()["ntrack"], o.tracks()["ntrack"])
    if s.cfg.shock:
        assert all(np.array_equal(a, b) for a, b in zip(g.active(hip.F_SHOCKED), o.active(oc.F_SHOCKED)))
    counts = g.regrid_counts()
    assert all(np.array_equal(a, b) for a, b in zip(counts, o.regrid_counts()))
    assert sum(a.sum() for a in counts) > 0
    assert g.time()[0][0] == o.t


@pytest.mark.gpu
@pytest.mark.parametrize("n", [6137, 6140, 8187, 12_003])
def test_gpu_regrid_blandford_mckee(n):
    """Cells and shock window on either side of a 2048-slot boundary of the chip-wide screen."""
    s = S.blandford_mckee_1d(n, lfac_shock=20., dth=5e-4 * 4000 / n)
    _equal(s, (1, 4))


@pytest.mark.gpu
@pytest.mark.parametrize("case", ["expanding", "expanding_circ", "box", "riemann", "jet"])
def test_gpu_regrid_other_rules(case):
    if case == "riemann":
        s = S.riemann_2d(11_000, 3, ly=3 / 11_000)
    elif case == "jet":                     # two dimensions, shock state cleared by the same launch
        s = S.bm_jet_2d(3, n_lo=400, n_hi=12_000)
    elif case == "box":
        s = S.reflecting_box(6000, mesh=1.)
    else:
        s = S.expanding_tube_1d(6000)
        if case == "expanding_circ":
            s = dataclasses.replace(s, cfg=s.cfg.replace(circ_regrid=1))
    _equal(s, (1, 35) if case == "riemann" else (1, 9))


@pytest.mark.gpu
@pytest.mark.parametrize("n", [1200, 1300, 1700])
def test_gpu_slot_scan_with_and_without_the_gradients(n):
    """Track lengths on either side of where the F1 slot scan gets a launch of its own."""
    s = S.riemann_2d(n, 9, ly=9 / n)
    g, o = hip.Grid(s), oc.OracleGrid(s)
    g.step(12)
    o.run(12)
    for f in (S.RHO, S.PPP, S.UU1, S.UU2, hip.F_X):
        assert np.array_equal(np.concatenate(g.active(f)), np.concatenate(o.active(f))), f


@pytest.mark.gpu
@pytest.mark.parametrize("n", [32_252, 32_253, 64_000])
def test_gpu_1d_time_step_of_many_tiles(n):
    """Track lengths (four ghost cells more) on either side of where the tiles' minima get a launch of their own."""
    s = S.shock_tube_1d(n)
    g, o = hip.Grid(s), oc.OracleGrid(s)
    g.step(5)
    o.run(5)
    for f in (S.RHO, S.PPP, S.UU1, hip.F_X):
        assert np.array_equal(g.active(f)[0], o.active(f)[0]), f
    assert g.time()[0][0] == o.t

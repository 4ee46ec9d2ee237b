"""The passes of a 1D step on tracks whose ghost cells, last cell or last face
fall on either side of a tile's end (a tile is 63 cells, ghost cells included),
and a grid loaded and stepped again after a state with other slots in use:
bit for bit the oracle's run."""
from __future__ import annotations

import numpy as np
import pytest

from gamma_amd import hip, setups as S
import oracle_ctypes as oc


def _equal(g, o, fields):
    for f in fields:
        a, b = np.concatenate(g.active(f)), np.concatenate(o.active(f))
        assert np.array_equal(a, b, equal_nan=True), f


@pytest.mark.gpu
@pytest.mark.parametrize("n", [8, 57, 58, 59, 60, 61, 120, 121, 122, 123, 185])
@pytest.mark.parametrize("kind", ["tube", "blast"])
def test_gpu_1d_tile_edges(n, kind):
    s = S.shock_tube_1d(n, geom=n % 2) if kind == "tube" else S.blandford_mckee_1d(n, lfac_shock=10.)
    g, o = hip.Grid(s), oc.OracleGrid(s)
    for k in (1, 24):                      # an odd and an even number of steps (plane swaps)
        g.step(k)
        o.run(k)
        _equal(g, o, (S.RHO, S.PPP, S.UU1, hip.F_X, hip.F_DX))
    assert g.time()[0][0] == o.t


@pytest.mark.gpu
def test_gpu_1d_restored_state_continues():
    """Saved after an odd number of steps, restored after others changed the track's length."""
    s = S.blandford_mckee_1d(400)
    g = hip.Grid(s)
    g.step(7)
    b = g.save_state()
    g.step(9)
    ref = {f: g.cells(f) for f in (S.RHO, S.PPP, S.UU1, hip.F_X)}
    g.step(30)
    g.restore_state(b)
    g.step(9)
    n = g.tracks()["ntrack"][0]
    for f, a in ref.items():
        assert np.array_equal(a[0, :n], g.cells(f)[0, :n])

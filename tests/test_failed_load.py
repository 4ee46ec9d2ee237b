"""A load that is refused leaves the grid as it was: it goes on with the tracks
it has, their hooks and the launches that suit them."""
from __future__ import annotations

import numpy as np
import pytest

from gamma_amd import hip, setups as S


def _check(lib_path, mk, steps):
    g, ref = hip.Grid(mk(), lib_path=lib_path), hip.Grid(mk(), lib_path=lib_path)
    g.step(3)
    s = mk()
    rc = s.cfg.replace(kin_mode=S.KIN_NONE, bnd_mode=S.BND_NONE, rg_mode=S.RG_NONE)
    n = g.cfg.ntracks_active
    for bad in (dict(ncell=s.cfg.ncell_mv + 1), dict(kin_mode=9), dict(rg_mode=7)):
        hooks = [hip.make_hooks(rc) for _ in range(n)]
        for k, v in bad.items():
            setattr(hooks[-1], k, v)
        arr = (hip.TrackHooks * n)(*hooks)
        assert g.L.gammahip_load(g.h, *[hip._p(a) for a in g._keep], arr, 0.) != 0
    g.step(steps)
    ref.step(3 + steps)
    assert np.array_equal(g.tracks()["ntrack"], ref.tracks()["ntrack"])
    for f in (S.RHO, S.PPP, S.UU1, hip.F_X):
        assert np.array_equal(g.cells(f), ref.cells(f), equal_nan=True), f


CASES = [(lambda: S.reflecting_box(32), 260),           # long enough for the blast to meet the user's walls
         (lambda: S.blandford_mckee_1d(200), 9), (lambda: S.riemann_2d_uneven(64, 8), 9)]


@pytest.mark.parametrize("mk,steps", CASES)
def test_emu_refused_load_changes_nothing(emu_lib, mk, steps):
    _check(emu_lib, mk, steps)


@pytest.mark.gpu
@pytest.mark.parametrize("mk,steps", CASES)
def test_gpu_refused_load_changes_nothing(mk, steps):
    _check(hip.LIB_PATH, mk, steps)

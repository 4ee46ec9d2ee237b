"""Slots past a track's end are left as they are by a step: a 1D step that
writes its result to a second set of planes shows the same values there, after
odd and even step counts alike, from a load, a restored state and the
particles' initialisation on."""
from __future__ import annotations

import dataclasses

import numpy as np
import pytest

from gamma_amd import hip, setups as S

FIELDS = (S.RHO, S.PPP, S.UU1, S.GMN, S.GMX, hip.F_DX)


def _unused(g, longest):
    return [g.cells(f)[0, longest:].copy() for f in FIELDS]


def _check(lib_path, regrid):
    s = S.blandford_mckee_1d(400)
    if not regrid:
        s = dataclasses.replace(s, cfg=s.cfg.replace(rg_mode=S.RG_NONE))
    g = hip.Grid(s, lib_path=lib_path)

    def hold(tell):
        longest = g.tracks()["ntrack"][0]
        ref = _unused(g, longest)
        for k in range(4):
            g.step(1)
            longest = max(longest, g.tracks()["ntrack"][0])
            for f, a, b in zip(FIELDS, ref, _unused(g, longest)):
                assert np.array_equal(a[len(a) - len(b):], b, equal_nan=True), (tell, f, k)

    hold("load")
    b = g.save_state()
    g.step(1)
    g.restore_state(b)
    hold("restored")
    g.apply(hip.INIT_GAMMAS)
    hold("INIT_GAMMAS")


@pytest.mark.parametrize("regrid", [True, False])
def test_emu_unused_slots_keep_their_values(emu_lib, regrid):
    _check(emu_lib, regrid)


@pytest.mark.gpu
@pytest.mark.parametrize("regrid", [True, False])
def test_gpu_unused_slots_keep_their_values(regrid):
    _check(hip.LIB_PATH, regrid)

"""The options that the library chooses by the grid (workgroup size, F1 sums
inside the update) can be given back to it, and the tuner starts from, compares
with and falls back to that choice."""
from __future__ import annotations

import numpy as np
import pytest

from gamma_amd import autotune, hip, setups as S
import oracle_ctypes as oc


class _Recorder:
    """A grid that notes the options set on it."""

    def __init__(self):
        self.opts = {}

    def set_options(self, **kw):
        self.opts.update(kw)

    def load_surrogate(self, w):
        pass


@pytest.mark.parametrize("form", ["DEFAULTS", "PLAIN"])
def test_tuner_starts_from_the_librarys_choice(form):
    g = _Recorder()
    autotune.apply(g, getattr(autotune, form))
    assert g.opts["block"] == "auto" and g.opts["f1fuse"] == "auto"
    space = dict(autotune.SPACE)
    assert "auto" in space["block"] and "auto" in space["f1fuse"]


def test_emu_auto_value_is_taken_and_checked(emu_lib):
    g = hip.Grid(S.riemann_2d(32, 8), lib_path=emu_lib)
    g.set_options(block=256, f1fuse=1)
    g.set_options(block="auto", f1fuse="auto")
    for bad in (-1, 4):
        assert g.L.gammahip_set_option(g.h, hip.OPT_AUTO, bad) != 0
    with pytest.raises(RuntimeError, match="block"):
        g.set_options(block=96)


@pytest.mark.gpu
def test_gpu_f1_sums_return_to_the_rule():
    """Ten fields: summed in the update unless asked otherwise (entry 4 of the
    kernel times counts the separate pass)."""
    g = hip.Grid(S.bm_jet_2d(12, 0.3, 40, 160))
    g.kernel_times()
    seen = []
    for opt in (None, 0, "auto", 1, "auto"):
        g.set_options(f1fuse=opt)
        g.step(2)
        seen.append(int(g.kernel_times()[1][4]))
    assert seen == [0, 6, 0, 0, 0]


def _separate_sums(lib_path):
    s = S.bm_jet_2d(12, 0.3, 40, 160)
    g, o = hip.Grid(s, lib_path=lib_path), oc.OracleGrid(s)
    g.set_options(block=128, f1fuse=0)
    g.step(30)
    o.run(30)
    for f in (S.RHO, S.PPP, S.UU1, S.UU2, S.GMX, hip.F_X):
        assert all(np.array_equal(a, b) for a, b in zip(g.active(f), o.active(f))), f


def test_emu_ten_fields_with_the_sums_in_a_pass_of_their_own(emu_lib):
    _separate_sums(emu_lib)


@pytest.mark.gpu
def test_gpu_ten_fields_with_the_sums_in_a_pass_of_their_own():
    _separate_sums(hip.LIB_PATH)


@pytest.mark.parametrize("setup,cand,idle", [
    (lambda: S.shock_tube_1d(32), {}, {"block", "remap", "occ", "f1fuse", "f1cell", "fuse"}),
    (lambda: S.shock_tube_1d(32), {"persist": 8}, {"f1fuse", "f1cell", "fuse"}),
    (lambda: S.shock_tube_1d(32), {"mlp_thr": 2}, {"f1fuse", "f1cell", "fuse"}),
    (lambda: S.reflecting_box(32), {}, {"f1fuse", "f1cell", "fuse"}),
    (lambda: S.ensemble_1d(4, sizes=(60, 80))[0], {}, {"block", "remap", "occ", "f1fuse", "f1cell", "fuse"}),
    (lambda: S.riemann_2d(32, 8), {}, set()),
])
def test_emu_tuner_leaves_out_options_without_effect(emu_lib, setup, cand, idle):
    g = hip.Grid(setup(), lib_path=emu_lib)
    cand = dict(autotune.PLAIN, **cand)
    assert {k for k, _ in autotune.SPACE if autotune.no_effect(g, k, cand)} == idle


def test_emu_tuner_times_nothing_without_effect(emu_lib):
    g = hip.Grid(S.shock_tube_1d(32), lib_path=emu_lib)
    r = autotune.tune(g, steps=1, settle=1, sweeps=1)
    for row in r["table"]:
        plain = row["persist"] == 0
        assert row["f1fuse"] == "auto" and row["f1cell"] == 0 and row["fuse"] == 0
        assert not plain or (row["block"] == "auto" and row["remap"] == 2 and row["occ"] == 0)
    assert {k: r["best"][k] for k in autotune.OPTION_KEYS}.keys() == autotune.DEFAULTS.keys()

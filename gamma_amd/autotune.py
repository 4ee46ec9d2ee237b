"""Autotuner for the launch options of the HIP backend.

Options: threads per workgroup of the per-cell kernels (the library's choice
for the grid, 64, 128, 256), XCD-aware tile order (off/on), two-step hipGraph
replay (off/on), persistent packed launch (off, or at most 4, 8, 16 or 32
workgroups per CU, each kernel's grid capped at what its registers and LDS let
a CU hold), the register-capped builds of the F1 face kernel and of the update
kernel (bit set, 0-3), the F1 flux sums inside the update kernel (the library's
choice, off, on), the fused F1 gradient-and-face pass (off/on), the cons2prim
solver (Brent, the reference's algorithm, or Newton) and, when a trained network
is given, the learned cons2prim start (off, or on with trigger exponents 2 and
4; Newton only).

Search: coordinate descent from the defaults -- each option in turn is set to
each of its values with the others held, the fastest kept -- repeated for
`sweeps` passes; options without effect on the grid (no_effect) are left out.  Each evaluation runs on the live grid (the production state,
not a toy): a short untimed run to settle (and capture the graph), then
`steps` timed steps between stream synchronisations.  The grid keeps evolving
while tuning, so the incumbent is re-timed with every challenger and the
comparison made within that pair.  The winner is applied to the grid and
returned with every evaluation made.
"""
from __future__ import annotations

import time

from . import setups as S

SPACE = (("solver", (0, 1)), ("block", ("auto", 64, 128, 256)), ("remap", (0, 1, 2)), ("graph", (0, 1)),
         ("persist", (0, 4, 8, 16, 32)), ("occ", (0, 1, 2, 3)), ("f1fuse", ("auto", 0, 1)), ("f1cell", (0, 1)), ("fuse", (0, 1, 2, 4)))
DEFAULTS = {"solver": 1, "block": "auto", "remap": 2, "graph": 0, "persist": 0, "occ": 0, "f1fuse": "auto",
            "f1cell": 0, "fuse": 0, "mlp_thr": None}
OPTION_KEYS = tuple(DEFAULTS)
# the plain form: the library's default launch with the reference's Brent solver
PLAIN = dict(DEFAULTS, solver=0)


def no_effect(grid, key: str, cand: dict) -> bool:
    """Whether an option changes nothing on this grid with the others as in
    cand: in 1D there are no F1 passes, and the five-launch step (all but
    packed launches, the learned start, Euler steps and user hooks) has launches
    of its own."""
    rc = grid.rc
    if rc.nd != 1:
        return False
    if key in ("f1fuse", "f1cell", "fuse"):
        return True
    if key not in ("block", "remap", "occ"):
        return False
    hooks = [h for h in grid.setup.hooks or [] if h]
    user = any(S.KIN_USER == h.get("kin_mode", rc.kin_mode) or S.BND_USER == h.get("bnd_mode", rc.bnd_mode)
               for h in hooks + [{}])
    return not (cand["persist"] or cand["mlp_thr"] is not None or rc.timestep == S.TS_EULER or rc.user_cell or user)


def apply(grid, cand: dict, surrogate=None):
    if cand.get("mlp_thr") is None and surrogate is not None:
        grid.load_surrogate(None)
    grid.set_options(solver=cand["solver"], block=cand["block"], remap=cand["remap"], graph=cand["graph"],
                     persist=cand["persist"], occ=cand["occ"], f1fuse=cand["f1fuse"], f1cell=cand["f1cell"],
                     fuse=cand["fuse"])
    if cand.get("mlp_thr") is not None:
        grid.load_surrogate(surrogate)
        grid.set_options(mlp_thr=cand["mlp_thr"])


def _time(grid, cand, surrogate, steps, settle):
    apply(grid, cand, surrogate)
    grid.step(settle)
    grid.sync()
    t0 = time.perf_counter()
    grid.step(steps)
    grid.sync()
    return 1e3 * (time.perf_counter() - t0) / steps


def tune(grid, steps: int = 6, settle: int = 2, sweeps: int = 2, surrogate=None,
         mlp_options=(None, 2, 4), margin: float = 0.005) -> dict:
    space = list(SPACE) + ([("mlp_thr", mlp_options)] if surrogate is not None else [])
    best = dict(DEFAULTS)
    table = []
    for _ in range(sweeps):
        for key, values in space:
            for v in values:
                if v == best[key] or no_effect(grid, key, best):
                    continue
                cand = dict(best, **{key: v})
                if cand["mlp_thr"] is not None and cand["solver"] != 1:
                    continue                     # the learned start seeds Newton only
                t_inc = _time(grid, best, surrogate, steps, settle)
                t_new = _time(grid, cand, surrogate, steps, settle)
                table.append(dict(cand, ms_per_step=round(t_new, 4), incumbent_ms=round(t_inc, 4)))
                if t_new < t_inc * (1. - margin):
                    best = cand
    # the pick must also beat the plain form on longer timings, taken in turn,
    # or the plain form stands: short timings differ by about 1 % from run to
    # run, as much as many of the options do
    t_best = t_plain = 0.
    for _ in range(2):
        t_best += _time(grid, best, surrogate, 2 * steps, settle)
        t_plain += _time(grid, PLAIN, surrogate, 2 * steps, settle)
    if not t_best < t_plain * (1. - margin):
        best = dict(PLAIN)
    ms = _time(grid, best, surrogate, steps, settle)
    return {"best": dict(best, ms_per_step=round(ms, 4)), "table": table}

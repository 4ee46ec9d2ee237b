"""The batch calls on host arrays go through staging buffers in chunks: counts
either side of a chunk, rows longer than three, an optional second start,
several threads at once and buffers given back between calls all return what
the states' own solves return."""
from __future__ import annotations

import threading

import numpy as np
import pytest

from gamma_amd import hip, surrogate as SG

G = 5. / 3.


def _case(n, seed):
    st = SG.synthetic_states(n, G, seed=seed, lf=(1., 30.), p_over_rho=(1e-6, 1e2))
    return st, SG.cold_guess(st, G)


def _equal(a, b):
    return all(np.array_equal(a[k], b[k]) for k in ("p", "iters", "fail", "used"))


@pytest.mark.gpu
@pytest.mark.parametrize("n", [1, 1000, 37_000, 40_000, 80_001])
@pytest.mark.parametrize("second", [False, True])
def test_gpu_batch_chunks(n, second):
    st, g = _case(n, 3)
    g2 = 1.1 * st[:, 3] if second else None
    a = SG.c2p_batch(st, g, G, guess2=g2)                       # rows of four
    b = SG.c2p_batch(st[:, :3].copy(), g, G, guess2=g2)         # rows of three
    assert _equal(a, b)
    for lo in range(0, n, 7_000):                               # one chunk each
        part = SG.c2p_batch(st[lo:lo + 7_000], g[lo:lo + 7_000], G, guess2=None if g2 is None else g2[lo:lo + 7_000])
        assert all(np.array_equal(a[k][lo:lo + 7_000], part[k]) for k in part)


@pytest.mark.gpu
def test_gpu_batch_threads_and_release():
    L = hip.load_library()
    cases = [_case(60_000 + 977 * k, k) for k in range(4)]
    ref = [SG.c2p_batch(st, g, G) for st, g in cases]
    assert L.gammahip_release_workspaces() == 0
    got = [None] * 4

    def work(k):
        for _ in range(3):
            got[k] = SG.c2p_batch(*cases[k], G)
            L.gammahip_release_workspaces()

    th = [threading.Thread(target=work, args=(k,)) for k in range(4)]
    [t.start() for t in th]
    [t.join() for t in th]
    assert all(_equal(a, b) for a, b in zip(ref, got))


def test_rows_are_taken_as_they_are_or_copied():
    st, _ = _case(50, 1)
    assert SG._rows(st) is st
    for other in (st[::2], st.astype(np.float32), np.asfortranarray(st), st[:, :3]):
        r = SG._rows(other)
        assert r.flags.c_contiguous and r.dtype == np.float64
        np.testing.assert_array_equal(r[:, :3], other[:, :3])

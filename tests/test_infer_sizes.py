"""Batch inference of device arrays in one launch, at counts either side of a
wavefront and a workgroup (FP32 path) and past one and two rounds of the
matrix-instruction path's 2048 workgroups of 256 states, whose walk over its
share reuses the network packed on chip: a state's answer has the bits it has
in a short batch.  The library keeps no device memory between calls (the
network is packed by each workgroup for itself)."""
from __future__ import annotations

import numpy as np
import pytest

from gamma_amd import hip, surrogate as SG
from test_zz_no_alloc import _Dev, _hip, _params

G53 = 5.0 / 3.0
ROUND = 2048 * 256


@pytest.mark.gpu
@pytest.mark.parametrize("mfma,n", [(0, 1), (0, 63), (0, 64), (0, 65), (0, 257), (0, 20_001),
                                    (1, ROUND), (1, ROUND + 3), (1, 2 * ROUND + 300)])
def test_gpu_inference_counts_in_one_launch(mfma, n):
    L, R = hip.load_library(), _hip()
    w = _params(5)
    st = np.ascontiguousarray(SG.synthetic_states(4999, G53, seed=17)[:, :3])     # odd: no period of a workgroup's
    ref = SG.infer(w, st, mfma=bool(mfma))
    reps = n // len(st) + 1
    big = np.ascontiguousarray(np.tile(st, (reps, 1))[:n])
    dw, ds, do = _Dev(R, w), _Dev(R, big), _Dev(R, np.full(n, np.nan))
    try:
        assert L.gammahip_mlp_infer_noalloc(dw.p, ds.p, n, do.p, mfma, None) == 0
        got = do.get(np.empty(n))              # a copy on the same (default) stream waits for the launch
    finally:
        for b in (dw, ds, do):
            b.free()
    want = np.tile(ref, reps)[:n]
    assert np.array_equal(got.view(np.uint64), want.view(np.uint64)), int(np.sum(got != want))

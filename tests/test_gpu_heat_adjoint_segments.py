"""The adjoint run from checkpoints gives what it gives with every state kept:
segments that end at, before and after a change of the time step and the light,
fixed-temperature and insulating boundaries, a mask, and the conduction
coefficients.  Both runs do the same operations in the same order, so the
fields agree bit for bit; the coefficients' sums are added by atomics in any
order: 23 steps of 1680 voxels and 6 neighbours, 2.3e5 terms, each addition
within 2^-53 of the largest partial sum (ten times the largest coefficient)."""
from __future__ import annotations

import numpy as np
import pytest

from test_gpu_heat_adjoint import case

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("every", [2, 4, 5, 7, 14, 15, 16, 20])
@pytest.mark.parametrize("bt", [0, 1])
def test_segments_equal_kept_states(bt, every):
    from mcmatlab_amd import api

    # checkpoints and a segment are fewer states than all of them, else those are kept
    assert -(-23 // every) + every + 1 < 24
    print(f"[adjoint-segments] bt {bt} every {every}", flush=True)
    T0, Om0, P, segs = case(bt, seed=21)  # 15 steps with the light on, 8 longer ones without
    assert T0.size == 1680 and sum(n for n, _, _ in segs) == 23
    mask = (np.arange(T0.size).reshape(T0.shape) % 3 == 0) | (np.asarray(P["M"]) == 3)
    kept = api.heat_adjoint(T0, Om0, P, segments=segs, targetMask=mask, coefGrad=True, maxStateBytes=1 << 30)
    cut = api.heat_adjoint(T0, Om0, P, segments=segs, targetMask=mask, coefGrad=True, checkpointEvery=every, maxStateBytes=0)
    assert kept["J"] == cut["J"] > 0
    for k in ("dJ_dQ", "dJ_dT0", "Omega"):
        assert np.array_equal(kept[k], cut[k]), k
    c = np.asarray(kept["dJ_dc"])
    assert np.max(np.abs(c - cut["dJ_dc"])) <= 2.3e5 * 2.0**-53 * np.max(np.abs(c)) * 10

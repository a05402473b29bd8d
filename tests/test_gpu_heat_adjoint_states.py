"""The adjoint with every state kept and with segments run again from
checkpoints: a field that does not vary along z has, in every layer, the
gradients of the one-layer problem.  The layers' states fit the memory kept for
them, the tall grid's (4.4 GB) do not."""
from __future__ import annotations

import numpy as np
import pytest

from test_gpu_heat_lines import line_case

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("every", [100, 261])
def test_segments_and_kept_states_agree(every):
    from mcmatlab_amd import api

    print(f"[adjoint-states] every {every}", flush=True)
    shape, nz, steps = (128, 125), 130, 264
    T1, Om1, P1 = line_case((*shape, 1), 0.05, seed=5, steps=steps, sinked=0)
    P1["dTdt_abs"] = P1["dTdt_abs"] * 0.05
    Pz = dict(P1)
    for k in ("M", "dTdt_abs"):
        Pz[k] = np.asfortranarray(np.repeat(P1[k], nz, axis=2))
    one = api.heat_adjoint(T1, Om1, P1, checkpointEvery=every)
    tall = api.heat_adjoint(np.asfortranarray(np.repeat(T1, nz, axis=2)), np.asfortranarray(np.repeat(Om1, nz, axis=2)), Pz,
                            checkpointEvery=every)
    # 264 steps of a few dozen FP64 roundings each, and the z solves of constant lines
    assert np.isfinite(one["J"]) and one["J"] > 0
    np.testing.assert_allclose(tall["J"], nz * one["J"], rtol=1e-10)
    for k in ("dJ_dQ", "dJ_dT0"):
        a, b = np.asarray(tall[k]), np.asarray(one[k])
        assert np.max(np.abs(a - b)) <= 1e-10 * np.max(np.abs(b)), k

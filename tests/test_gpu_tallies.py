"""The raw tallies of a run on a stream of its own are those that normalize()
forms the fluence from: the absorbed weight over V mua N, rounded to single."""
from __future__ import annotations

import numpy as np
import pytest

import models

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("copies", [1, 8])
@pytest.mark.parametrize("shape", [(13, 18, 27), (40, 1, 9)])  # ragged bricks, linear order
def test_tallies_are_complete_and_linear(shape, copies):
    import torch

    from mcmatlab_amd import api

    print(f"[gpu-tallies] {shape} {copies}", flush=True)
    n = 100000
    m = models.base(n=27)
    m.MC.M = np.asfortranarray(np.random.default_rng(1).integers(1, 5, shape).astype(np.uint8))
    plan = api.MCPlan(m)
    try:
        plan.set_fluence_copies(copies)
        stream = torch.cuda.Stream()
        plan.simulate(n, seed=5, stream=stream.cuda_stream)
        ptr, launched = plan.tallies()
        assert launched == n

        class View:
            __cuda_array_interface__ = {"shape": (int(np.prod(shape)),), "typestr": "<f8", "data": (ptr, False), "version": 2}

        D = torch.as_tensor(View(), device="cuda").cpu().numpy().reshape(shape, order="F")
        F = np.asarray(plan.normalize()["NFR"]).reshape(shape, order="F")
    finally:
        plan.close()
    mua = np.asarray(m.MC.mediaProperties["mua"]).ravel()[m.MC.M.astype(int) - 1]
    assert D.sum() > 0
    np.testing.assert_allclose(F, D / (m.G.dx * m.G.dy * m.G.dz * n * mua), rtol=2.0**-23)

"""The raw tallies of a run on a stream of its own are those that normalize()
forms the fluence from: the absorbed weight over V mua N, rounded to single."""
from __future__ import annotations

import ctypes as C

import numpy as np
import pytest

import models

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("copies", [1, 8])
@pytest.mark.parametrize("shape", [(13, 18, 27), (40, 1, 9)])  # ragged bricks, linear order
def test_tallies_are_complete_and_linear(shape, copies):
    from mcmatlab_amd import _lib, api

    print(f"[gpu-tallies] {shape} {copies}", flush=True)
    hip = _lib.lib()  # (the runtime that the library itself uses, whatever else is loaded)
    n = 100000
    m = models.base(n=27)
    m.MC.M = np.asfortranarray(np.random.default_rng(1).integers(1, 5, shape).astype(np.uint8))
    plan = api.MCPlan(m)
    stream = C.c_void_p()
    assert hip.hipStreamCreateWithFlags(C.byref(stream), 1) == 0  # hipStreamNonBlocking
    try:
        plan.set_fluence_copies(copies)
        plan.simulate(n, seed=5, stream=stream)
        ptr, launched = plan.tallies()
        assert launched == n
        D = np.empty(int(np.prod(shape)))
        assert hip.hipMemcpy(C.c_void_p(D.ctypes.data), C.c_void_p(ptr), C.c_size_t(D.nbytes), 2) == 0  # device to host
        D = D.reshape(shape, order="F")
        F = np.asarray(plan.normalize()["NFR"]).reshape(shape, order="F")
    finally:
        plan.close()
        assert hip.hipStreamDestroy(stream) == 0
    mua = np.asarray(m.MC.mediaProperties["mua"]).ravel()[m.MC.M.astype(int) - 1]
    assert D.sum() > 0
    np.testing.assert_allclose(F, D / (m.G.dx * m.G.dy * m.G.dz * n * mua), rtol=2.0**-23)

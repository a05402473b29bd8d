"""Downloads of large arrays through pinned blocks: a state that was not
advanced comes back as it was sent, bit for bit, for sizes below, at and above
those where the staged copy starts, in whole and partial blocks and stripes."""
from __future__ import annotations

import numpy as np
import pytest

from test_gpu_heat_lines import line_case

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape", [(5, 4, 3), (64, 64, 128), (128, 128, 128), (131, 127, 127), (128, 256, 65), (257, 129, 129)])
def test_state_comes_back(shape):
    from mcmatlab_amd import api

    print(f"[downloads] {shape}", flush=True)
    _, _, P = line_case(shape, 0.05, steps=0)
    rng = np.random.default_rng(shape[0])
    T = np.asfortranarray(rng.uniform(20, 90, shape).astype(np.float32))
    Om = np.asfortranarray(rng.uniform(0, 2, shape).astype(np.float32))
    plan = api.HeatPlan(T, Om, P, precision="fp64", scheme="dgadi")
    try:
        for f64 in (True, False):
            r = plan.download(f64=f64)
            assert np.array_equal(r["T"], T) and np.array_equal(r["Omega"], Om)
            if f64:
                assert np.array_equal(r["T_f64"], T.astype(np.float64)) and np.array_equal(r["Omega_f64"], Om.astype(np.float64))
    finally:
        plan.close()

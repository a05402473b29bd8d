"""Values at the limits of what the heat steps are given: temperatures without a
finite reciprocal, and coefficients without a value where none is needed."""
from __future__ import annotations

import numpy as np
import pytest

from test_gpu_heat_lines import line_case

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape", [(6, 5, 7), (6, 5, 600)])  # lines in registers, a lane a line
@pytest.mark.parametrize("scheme", ["dgadi", "explicit"])
def test_damage_at_infinite_and_zero_absolute_temperature(scheme, shape):
    """A exp(-E / (R T)) has the limits A for T -> inf and 0 for T -> 0.  The
    corners of a grid with fixed boundaries keep their temperature and touch
    fixed voxels only."""
    from mcmatlab_amd import api

    print(f"[heat-limits] {scheme} {shape}", flush=True)
    T0, Om0, P = line_case(shape, 0.05, nM=2, steps=3, sinked=1)
    P["M"][:] = 0
    P["A"], P["E"] = np.array([2.0, 3.0]), np.array([5e3, 5e3])
    T = T0.astype(np.float64)
    corners = {(0, 0, 0): (np.inf, 2.0), (0, -1, 0): (-np.inf, 2.0), (-1, 0, 0): (-273.15, 0.0), (-1, -1, -1): (np.nan, np.nan)}
    for at, (t, _) in corners.items():
        T[at] = t
    api.finiteElementHeatPropagator(T0, Om0, P, precision="fp64", scheme=scheme, state_f64=(T, np.zeros(shape)))
    T64, Om64 = api.finiteElementHeatPropagator.last_state
    rest = np.ones(shape, bool)
    for at, (t, rate) in corners.items():
        np.testing.assert_equal(T64[at], t)
        np.testing.assert_allclose(Om64[at], 3 * 0.05 * rate, rtol=1e-14)
        rest[at] = False
    assert np.all(np.isfinite(T64[rest])) and np.all(np.isfinite(Om64[rest])) and np.all(Om64[rest] > 0)

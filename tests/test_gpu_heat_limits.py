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


@pytest.mark.parametrize("precision,scheme", [("fp64", "dgadi"), ("fp64", "explicit"), ("fp32", "dgadi"), ("fp32", "explicit")])
@pytest.mark.parametrize("shape", [(70, 1, 9), (1, 20, 9), (9, 20, 1), (1, 1, 33), (66, 7, 6)])
def test_coefficients_of_pairs_that_never_meet_are_not_used(precision, scheme, shape):
    """An axis of one voxel has no neighbours, and media laid in layers of one
    voxel never meet themselves: whatever their coefficients are, 0, infinite or
    no number, the state is the same."""
    from mcmatlab_amd import api

    print(f"[heat-limits] {precision} {scheme} {shape}", flush=True)
    T0, Om0, P = line_case(shape, 0.05, nM=4, steps=6, sinked=0)
    M = np.zeros(shape, np.uint8)
    M[:] = (np.arange(shape[2]) % 3)[None, None, :]  # medium 3 nowhere
    if shape[0] > 2:
        M[-1] = 0  # more pairs along x and z
    P["M"] = np.asfortranarray(M)
    met = np.zeros((4, 4, 3), bool)
    for d in range(3):
        lo, hi = (np.moveaxis(M, d, 0)[s].ravel() for s in (slice(None, -1), slice(1, None)))
        met[lo, hi, d] = met[hi, lo, d] = True
    assert not met.all()
    r = []
    for value in (0.0, np.inf, np.nan):
        c = np.array(P["dTdtperdeltaT"], copy=True)
        c[~met] = value
        T, Om, _, mx = api.finiteElementHeatPropagator(T0, Om0, dict(P, dTdtperdeltaT=c), precision=precision, scheme=scheme)
        assert np.all(np.isfinite(T)) and np.all(np.isfinite(Om))
        r.append((T, Om, mx))
    for other in r[1:]:
        for a, b in zip(r[0], other):
            assert np.array_equal(a, b)

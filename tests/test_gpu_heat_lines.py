"""FP64 DG-ADI line solves at the edges of the compiled line shapes and at time
steps below and above the explicit limit (no to all reduction steps of the line
solver), against the FP64 oracle."""
from __future__ import annotations

import numpy as np
import pytest

import oracle_lib as OL

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def api():
    from mcmatlab_amd import _lib, api as A

    assert _lib.lib().mcm_device_count() >= 1
    return A


def line_case(shape, dt, nM=5, seed=0, steps=3, sinked=1):
    """Random media (runs of a few voxels), coefficients of about 1 / s per axis."""
    rng = np.random.default_rng(seed)
    M = np.repeat(rng.integers(0, nM, size=(shape[0], shape[1], (shape[2] + 2) // 3)), 3, axis=2)[:, :, :shape[2]].astype(np.uint8)
    P = {"M": np.asfortranarray(M), "A": np.where(np.arange(nM) % 2, 1e10, 0.0), "E": np.where(np.arange(nM) % 2, 7e4, 0.0),
         "dTdtperdeltaT": rng.uniform(0.2, 2.0, (nM, nM, 3)).astype(np.float32),
         "dTdt_abs": np.asfortranarray(rng.uniform(0, 5, shape).astype(np.float32)), "useAllCPUs": False, "heatBoundaryType": sinked,
         "tempSensorCornerIdxs": np.zeros(0), "tempSensorInterpWeights": np.zeros((0, 3)), "lightsOn": True, "steps": steps, "dt": dt}
    T0 = np.asfortranarray((37 + 8 * rng.random(shape)).astype(np.float32))
    return T0, np.zeros(shape, np.float32, order="F"), P


# the largest off-diagonal / diagonal ratio is about dt / (1 + 2 dt): 0.05 (no
# or one reduction step) and 0.45 (most or all).  Rounding: eps * condition
# number (4 dt) * a few operations per row * 3 steps of 3 solves, far below
# 4e-12 of the field's largest value.  (Not dt >> 5: with insulated boundaries
# and a source such steps overshoot by orders of magnitude, and the oracle's
# own rounding exceeds any useful bound.)
@pytest.mark.parametrize("dt", [0.05, 5.0])
@pytest.mark.parametrize("n", [1, 2, 31, 33, 64, 97, 128, 161, 208, 209, 256, 257, 417, 512])
@pytest.mark.parametrize("axis", [0, 1, 2])
def test_line_shapes_and_time_steps(api, axis, n, dt):
    shape = [17, 3, 4]
    shape[axis] = n
    if axis != 0:
        shape[0] = 18  # a full and a partly filled group of 16 lines
    T0, Om0, P = line_case(tuple(shape), dt, seed=n, sinked=n % 2)
    print(f"[gpu-heat-lines] {shape} dt {dt}", flush=True)
    api.finiteElementHeatPropagator(T0, Om0, P, precision="fp64")
    T64, _ = api.finiteElementHeatPropagator.last_state
    ref = OL.oracle_heat(T0, Om0, P, variant=OL.HEAT_FP64_DGADI)
    assert np.max(np.abs(T64 - ref["T_f64"])) <= 4e-12 * np.max(np.abs(ref["T_f64"]))


def test_many_media_read_coefficients_from_memory(api):
    """23 media: the coefficient tables no longer fit the kernels' LDS copies."""
    T0, Om0, P = line_case((35, 21, 40), 0.05, nM=23, seed=3)
    api.finiteElementHeatPropagator(T0, Om0, P, precision="fp64")
    T64, Om64 = api.finiteElementHeatPropagator.last_state
    ref = OL.oracle_heat(T0, Om0, P, variant=OL.HEAT_FP64_DGADI)
    assert np.max(np.abs(T64 / ref["T_f64"] - 1)) <= 4e-12
    np.testing.assert_allclose(Om64, ref["Omega_f64"], rtol=1e-9, atol=0)


# the FP32 sweeps repeat the reference's operations one by one: same bits as the
# oracle but for the damage's exp
@pytest.mark.parametrize("steps", [2, 6])  # without and with the line factors
@pytest.mark.parametrize("n", [1, 2, 3, 103, 104, 106, 210, 211, 420, 421])
@pytest.mark.parametrize("axis", [0, 1, 2])
def test_fp32_line_lengths(api, axis, n, steps):
    shape = [17, 3, 4]
    shape[axis] = n
    if axis != 0:
        shape[0] = 35  # a full and a partly filled group of 32, 16 or 8 lines
    T0, Om0, P = line_case(tuple(shape), 0.3, seed=n, steps=steps, sinked=n % 2)
    print(f"[gpu-heat-lines32] {shape} steps {steps}", flush=True)
    T, Om, _, mx = api.finiteElementHeatPropagator(T0, Om0, P, precision="fp32")
    ref = OL.oracle_heat(T0, Om0, P, variant=OL.HEAT_FP32_DGADI)
    np.testing.assert_array_equal(T, ref["T"])
    np.testing.assert_array_equal(mx, ref["maxMediaTemps"])
    np.testing.assert_allclose(Om, ref["Omega"], rtol=1e-5)


def test_fp32_factors_follow_the_time_step(api):
    """Runs of alternating time steps and lengths, replayed graphs and a group:
    the line factors in memory are always those of the run's own dt."""
    T0, Om0, P = line_case((35, 21, 18), 0.3, steps=1)
    runs = [(8, 0.3, 1), (8, 0.1, 0), (8, 0.3, 1), (2, 0.1, 0), (2, 0.3, 1), (8, 0.1, 0)]
    plain = api.HeatPlan(T0, Om0, P, precision="fp32", graph_steps=0)
    graphs = api.HeatPlan(T0, Om0, P, precision="fp32", graph_steps=2)
    grouped = api.HeatPlan(T0, Om0, P, precision="fp32", graph_steps=0)
    other = api.HeatPlan(T0, Om0, P, precision="fp64", graph_steps=0)
    group = api.HeatGroup([grouped, other], steps_per_graph=2)
    T, Om = T0, Om0
    for steps, dt, on in runs:
        for _ in range(steps):  # one step a call: never factored
            plain.advance(1, dt, on)
        graphs.advance(steps, dt, on)
        group.advance(steps, [dt, dt], [on, on])
        Pr = dict(P, steps=steps, dt=dt, lightsOn=bool(on))
        ref = OL.oracle_heat(T, Om, Pr, variant=OL.HEAT_FP32_DGADI)
        T, Om = ref["T"], ref["Omega"]
        for plan in (plain, graphs, grouped):
            np.testing.assert_array_equal(plan.download(f64=False)["T"], T)
    group.close()
    for plan in (plain, graphs, grouped, other):
        plan.close()

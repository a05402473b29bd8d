"""FP32 DG-ADI lines on both sides of each change of kernel.  A workgroup takes 32,
16 or 8 lines whose pitch (the odd number n or n + 1) times four numbers fits into
54 KB; longer lines take a lane each.  The sweeps repeat the reference's
operations one by one: the same bits as the oracle but for the damage's exp."""
from __future__ import annotations

import numpy as np
import pytest

import oracle_lib as OL
from test_gpu_heat_lines import line_case

pytestmark = pytest.mark.gpu

LAST = [max(n for n in range(1, 1000) if lines * (n | 1) <= 54 * 1024 // 16) for lines in (32, 16, 8)]


def test_the_last_lengths_are_those_of_the_kernels_comment():
    assert LAST == [107, 215, 431]


def check(shape, steps, sinked, seed):
    from mcmatlab_amd import api

    print(f"[gpu-heat-lines32] {shape} steps {steps} sinked {sinked}", flush=True)
    T0, Om0, P = line_case(tuple(shape), 0.3, seed=seed, steps=steps, sinked=sinked)
    T, Om, _, mx = api.finiteElementHeatPropagator(T0, Om0, P, precision="fp32")
    ref = OL.oracle_heat(T0, Om0, P, variant=OL.HEAT_FP32_DGADI)
    np.testing.assert_array_equal(T, ref["T"])
    np.testing.assert_array_equal(mx, ref["maxMediaTemps"])
    np.testing.assert_allclose(Om, ref["Omega"], rtol=1e-5)


@pytest.mark.parametrize("sinked", [0, 1])
@pytest.mark.parametrize("steps", [2, 6])  # without and with the line factors
@pytest.mark.parametrize("n", sorted({*LAST, *(n + 1 for n in LAST), 600}))
@pytest.mark.parametrize("axis", [0, 1, 2])
def test_line_lengths_around_each_change(axis, n, steps, sinked):
    shape = [35, 5, 4]  # y and z lines: a full and a partly filled group
    shape[axis] = n
    check(shape, steps, sinked, seed=n)


@pytest.mark.parametrize("shape", [(600, 108, 5), (33, 600, 216), (432, 4, 431), (500, 3, 700)])
def test_axes_of_different_kernels(shape):
    """Axes too long for LDS, without factors, beside factored ones."""
    check(shape, 6, 1, seed=sum(shape))

"""Voxel order, parked deposits and launch shapes of the transport kernel.

A packet of a pure absorber stays in its column, so the fluence is known in
every voxel: the closed form checks where each deposit goes for whole and
ragged 4 x 4 x 4 bricks and for the thin grids that stay in linear order.
The packets of a run and their trajectories do not depend on how a run is cut
into launches or items, so runs cut in different ways give the same counters
and the same sums up to the order of the FP64 additions (1e-13 relative),
rounded to single: 2^-23 relative."""
from __future__ import annotations

import numpy as np
import pytest

import models
from mcmatlab_amd.model import media_table

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def api():
    from mcmatlab_amd import _lib, api as A

    assert _lib.lib().mcm_device_count() >= 1
    return A


def same(a, b):
    for k in a:
        x, y = np.asarray(a[k], np.float64), np.asarray(b[k], np.float64)
        if x.dtype.kind == "f" and x.ndim:
            np.testing.assert_allclose(x, y, rtol=2.0**-23, atol=0, err_msg=k)


SHAPES = [(4, 4, 4), (8, 12, 4), (5, 7, 9), (13, 4, 66), (1, 60, 3), (3, 3, 3), (2, 2, 40), (17, 1, 5)]


@pytest.mark.parametrize("shape", SHAPES)
def test_fluence_of_a_pure_absorber_by_column(api, shape):
    print(f"[mc-order] absorber {shape}", flush=True)
    nx, ny, nz = shape
    d, N = 0.01, 1000
    rng = np.random.default_rng(nx * 10007 + ny * 101 + nz)
    mua = np.array([3.0, 0.5, 8.0, 1.0])
    m = models.base(n=4)
    m.G.dx = m.G.dy = m.G.dz = d
    m.MC.M = np.asfortranarray(rng.integers(1, 5, shape).astype(np.uint8))
    m.MC.mediaProperties = media_table(mua, np.full(4, 1e-8), np.full(4, 0.9), np.ones(4))
    for ix, iy in {(0, 0), (nx - 1, ny - 1), (nx // 2, ny // 3)}:
        # off the voxel's centre: positions on voxel boundaries are ambiguous
        m.MC.lightSource.xFocus = float((ix - nx / 2 + 0.45) * d)
        m.MC.lightSource.yFocus = float((iy - ny / 2 + 0.45) * d)
        plan = api.MCPlan(m)
        try:
            plan.simulate(N, seed=3)
            assert plan.counters()["substeps"] == N * nz
            F = np.asarray(plan.normalize()["NFR"], np.float64).reshape(shape, order="F")
        finally:
            plan.close()
        a = mua[m.MC.M[ix, iy] - 1]
        w = np.exp(-d * np.concatenate([[0.0], np.cumsum(a)[:-1]]))
        expect = w * -np.expm1(-a * d) / (a * d**3)
        # a sub-step rounds the length, the exponential (2 ulp), two products and
        # the difference in single precision: 6 roundings of the weight each
        np.testing.assert_allclose(F[ix, iy], expect, rtol=(6 * nz + 4) * 2.0**-24)
        F[ix, iy] = 0
        assert not F.any()


@pytest.mark.parametrize("name,n,cut", [
    ("pencil_bt1", 1, 1), ("pencil_bt1", 65, 64), ("pencil_bt3", 1025, 17), ("fresnel_bt1", 20000, 1030), ("planewave_bt2", 70001, 65536),
    ("criteria_scatter", 66, 65), ("criteria_collected", 5000, 1023), ("criteria_now", 5000, 64),
    ("pencil_bt1", 300000, 299999)])
def test_cutting_a_run_changes_nothing(api, name, n, cut):
    """Launches that leave lanes empty, fill one wavefront or one workgroup per
    CU, or fill the chip."""
    print(f"[mc-order] {name} {n} {cut}", flush=True)
    m = models.cases()[name]()
    r = []
    for ends in ([n], [cut, n], [cut // 2, cut, n]):
        plan = api.MCPlan(m)
        try:
            first = 0
            for end in ends:
                if end > first:
                    plan.simulate(end - first, seed=8, firstPhoton=first)
                    first = end
            c = plan.counters()
            r.append((c, plan.normalize()))
        finally:
            plan.close()
    for c, o in r[1:]:
        assert {k: c[k] for k in c} == {k: r[0][0][k] for k in c}
        same(r[0][1], o)


@pytest.mark.parametrize("kind", ["batch", "multi"])
def test_as_many_items_and_media_as_fit(api, kind):
    """256 items of 8 media: the largest tables in LDS."""
    print(f"[mc-order] {kind}", flush=True)
    m = models.base(n=9)
    mp = media_table(np.linspace(0.5, 20, 8), np.linspace(50, 200, 8), np.full(8, 0.9), np.ones(8))
    m.MC.mediaProperties = mp
    m.MC.M = np.asfortranarray(np.random.default_rng(2).integers(1, 9, (9, 9, 9)).astype(np.uint8))
    plan = api.MCPlan(m)
    try:
        items = [(0, 37 + i, 100 + i, 0) for i in range(256)]
        got = plan.batch(items) if kind == "batch" else api.multi_run([plan], [(0, *it) for it in items])
        for i in (0, 1, 127, 254, 255):
            plan.simulate(items[i][1], seed=items[i][2])
            ref = plan.normalize()
            a, b = np.asarray(got[i]["NFR"], np.float64).ravel(order="F"), np.asarray(ref["NFR"], np.float64).ravel(order="F")
            np.testing.assert_allclose(a, b, rtol=2.0**-23, atol=0)
    finally:
        plan.close()


def test_gradient_run_of_more_packets_than_one_launch_takes(api):
    """2^22 packets fill a launch's records; the rest of the run counts as much."""
    m = models.base(n=6)
    n, box = 3 << 21, ((1, 5), (1, 5), (2, 6))
    plan = api.MCPlan(m)
    try:
        r = plan.absorbed_power(box, n, seed=4, grad=False)
        plan.simulate(n, seed=4)
        F = np.asarray(plan.normalize()["NFR"], np.float64).reshape(6, 6, 6, order="F")
        mua = m.MC.mediaProperties["mua"].ravel()
    finally:
        plan.close()
    V = m.G.dx * m.G.dy * m.G.dz
    P = (F * mua[m.MC.M.astype(int) - 1] * V)[1:5, 1:5, 2:6].sum()
    # the same packets: their paths differ only where the two kernels round differently
    assert abs(r["J"] - P) <= 5 * r["J_se"]

"""Binning of more sets than the workgroups of a pass take in one round, bit for
bit against the oracle; few distinct values, so that equal distances are spread
over rounds and workgroups."""
from __future__ import annotations

import numpy as np
import pytest

import oracle_lib as OL
from test_gpu_binning import same

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n1", [1024 * 2048 - 1, 1024 * 2048 + 1, 4500001])
def test_rounds(n1):
    from mcmatlab_amd import api

    print(f"[gpu-binning] rounds {n1}", flush=True)
    rng = np.random.default_rng(n1)
    pv = np.asfortranarray(rng.integers(1, 40, (3, n1)).astype(np.float32) / np.float32(7))
    o, b = api.getDownsampledParamVals(pv, 12)
    ro, rb = OL.oracle_binning(pv, 12)
    assert same(o, ro) and same(b, rb)

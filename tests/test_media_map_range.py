"""A media map may hold 1..nM only, for every number of media up to 256."""
import ctypes as C
import os

import numpy as np
import pytest

import models
from mcmatlab_amd import _lib, abi
from mcmatlab_amd.model import media_table

pytestmark = pytest.mark.skipif(not os.path.exists(_lib.LIB_PATH), reason="libmcm.so not built")


@pytest.mark.parametrize("nM", [1, 2, 255, 256])
@pytest.mark.parametrize("last", [False, True])
def test_media_outside_the_table_are_refused(nM, last):
    m = models.base(n=4)
    m.MC.mediaProperties = media_table(np.full(nM, 1.0), np.full(nM, 10.0), np.full(nM, 0.9), np.ones(nM))
    sz = abi.mcm_mc_sizes()
    for v in (0, 1, min(nM, 255), nM + 1):
        if v > 255:
            continue
        M = np.ones((4, 4, 4), np.uint8, order="F")
        M[(-1, -1, -1) if last else (0, 0, 0)] = v
        m.MC.M = M
        inp = abi.MCInputs(m, seed=1)
        rc = _lib.lib().mcm_mc_output_sizes(C.byref(inp.struct), C.byref(sz))
        assert rc == (abi.MCM_OK if 1 <= v <= nM else abi.MCM_ERR_INVALID_ARGUMENT), v

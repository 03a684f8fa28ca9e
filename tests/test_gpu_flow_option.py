"""The "flow" option of a handle: -1 leaves the kind of sweep to the matrix's size."""
import numpy as np
import pytest

import race_amd as R
from race_amd import matgen as M

pytestmark = pytest.mark.gpu


def test_automatic_choice_can_be_set_again():
    rp, col = M.stencil27(12)
    n = len(rp) - 1
    ce = R.Interface(n, 64, R.ONE, rp, col, symm_hint=True)
    ce.RACEColor()
    prp, pcol, pval = M.make_diag_first(*M.permute(rp, col, M.gs_values(rp, col, 1), ce.getPerm(), ce.getInvPerm()))
    launches = []
    for flow in (None, 0, -1, 1, -1):
        if flow is not None:
            ce.setOption("flow", flow)
        dx, db = R.DeviceArray.from_host(np.zeros(n)), R.DeviceArray.from_host(np.ones(n))
        launches.append(ce.launchCount(ce.registerDevice(R.K_GS, prp, pcol, pval, dx, db)))
    assert launches[0] == launches[2] == launches[3] == launches[4] == 1 and launches[1] > 1
    for bad in (-2, 2):
        with pytest.raises(Exception):
            ce.setOption("flow", bad)

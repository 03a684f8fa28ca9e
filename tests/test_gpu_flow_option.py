"""The "flow" option of a handle: -1 leaves the kind of sweep to the matrix's size;
automatic sweeps on many streams."""
import numpy as np
import pytest

import race_amd as R
from race_amd import _lib as L
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


def test_more_streams_than_state_sets():
    """ten streams, each with vectors of its own: eight sweep in one launch, the
    others by phases, all with the bits of synchronous phase launches"""
    rp, col = M.stencil27(12)
    n = len(rp) - 1
    owners = []
    for _ in range(10):
        owners.append(R.Interface(n, 64, R.ONE, rp, col, symm_hint=True))
    ce = owners[0]
    ce.RACEColor()
    mat = M.make_diag_first(*M.permute(rp, col, M.gs_values(rp, col, 1), ce.getPerm(), ce.getInvPerm()))
    bs = [M.uniform_vec(n, k) for k in range(len(owners))]
    vecs = [(R.DeviceArray.from_host(np.zeros(n)), R.DeviceArray.from_host(b)) for b in bs]
    fid = ce.registerDevice(R.K_GS, *mat, *vecs[0])
    assert ce.launchCount(fid) == 1
    for _ in range(6):
        for k, o in enumerate(owners):
            ce.setVectors(fid, *vecs[k])
            ce.executeAsync(fid, False, stream=o.stream())
            ce.executeAsync(fid, True, stream=o.stream())
    assert L.load().race_device_synchronize() == 0
    assert ce.flowAborts(fid) == 0
    ce.setOption("flow", 0)
    dx, db = R.DeviceArray.from_host(np.zeros(n)), R.DeviceArray.from_host(bs[0])
    ref = ce.registerDevice(R.K_GS, *mat, dx, db)
    for k in range(len(owners)):
        dx.upload(np.zeros(n))
        db.upload(bs[k])
        for _ in range(6):
            ce.executeFunction(ref, False)
            ce.executeFunction(ref, True)
        assert np.array_equal(vecs[k][0].download(), dx.download()), k

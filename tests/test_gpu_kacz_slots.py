"""The Kaczmarz kernels that hold fewer column ids: sweeps with more chains than
find a place at once, and batches that keep the chip busy for several times
their longest chain path.  The arithmetic is that of the other kernels, so the
results are the same bits; and against the oracle in RACE order."""
import numpy as np
import pytest

import race_amd as R
from race_amd import matgen as M

from .conftest import relerr

pytestmark = pytest.mark.gpu

# a column is written by at most ten rows of up to a hundred products each
TOL = {R.FP64: 1e-12, R.FP32: 2e-5}


def _dt(prec):
    return np.float64 if prec == R.FP64 else np.float32


def _calls(ce, rev):
    """the schedule's leaves in order, as the oracle takes them (a reverse leaf
    runs from hi - 1 down to lo)"""
    _, lo, hi = ce.schedule(rev)
    return np.stack([hi - 1, lo - 1] if rev else [lo, hi], axis=1).reshape(-1)


def _prep(rp, col, val, T):
    ce = R.Interface(len(rp) - 1, T, R.TWO, rp, col, symm_hint=True)
    ce.RACEColor()
    return (ce,) + M.make_diag_first(*M.permute(rp, col, val, ce.getPerm(), ce.getInvPerm()))


# 7-point: 16 right-hand sides, about 2600 chains at once; 27-point: 2000
@pytest.mark.parametrize("prec", [R.FP64, R.FP32])
@pytest.mark.parametrize("stencil,g,T,nrhs", [(M.stencil7, 64, 1024, 16), (M.stencil27, 80, 2048, 8)])
def test_many_chains_at_once(oracle, stencil, g, T, nrhs, prec):
    rp, col = stencil(g)
    n = len(rp) - 1
    ce, prp, pcol, pval = _prep(rp, col, M.gs_values(rp, col, 5), T)
    b = M.uniform_vec(n, 6, nrhs=nrhs).astype(_dt(prec))
    xs = []
    for flow in (0, 1):
        ce.setOption("flow", flow)
        dx, db = R.DeviceArray.from_host(np.zeros(n * nrhs, _dt(prec))), R.DeviceArray.from_host(b)
        fid = ce.registerDevice(R.K_KACZ, prp, pcol, pval, dx, db, nrhs=nrhs, val_precision=prec, vec_precision=prec)
        for rev in (False, True):
            print("case many chains", g, prec, flow, rev, flush=True)
            ce.executeFunction(fid, rev)
        assert ce.flowAborts(fid) == 0
        xs.append(dx.download())
    assert np.array_equal(xs[0], xs[1])
    # the first right-hand side in the colouring's order
    xo = np.zeros(n)
    for rev in (False, True):
        oracle.run_calls(oracle.K_KACZ, prp, pcol, pval, xo, b[:n].astype(np.float64), _calls(ce, rev))
    assert relerr(xs[0][:n].astype(np.float64), xo) <= TOL[prec]


@pytest.mark.parametrize("prec", [R.FP64, R.FP32])
@pytest.mark.parametrize("bs", [256, 512, 1024])
def test_busy_batch(oracle, bs, prec):
    """8 right-hand sides of 1024 banded matrices and graphs of about one size:
    the work is about 1024 * 8 / (256 CUs * 4 workgroups) = 8 times a path"""
    nrhs, dt = 8, _dt(prec)
    batch = R.Batch(R.K_KACZ, prec, prec, nrhs=nrhs)
    keep = []
    mats = [_prep(*m[3:], T=4) for m in M.batch_matrices(16, 4, 500, 700)]
    rp, col = M.stencil7(8)
    mats.append(_prep(rp, col, M.gs_values(rp, col, 2), 4))
    for k in range(1024):
        ce, prp, pcol, pval = mats[k % len(mats)]
        b = M.uniform_vec(len(prp) - 1, 90 + k, nrhs=nrhs).astype(dt)
        dx, db = R.DeviceArray.from_host(np.zeros(len(b), dt)), R.DeviceArray.from_host(b)
        batch.add(ce, prp, pcol, pval, dx, db)
        keep.append((k % len(mats), dx, b))
    for key, v in (("bundle_threads", bs), ("bundle_rows", 128), ("flow", 1)):
        batch.setOption(key, v)
    batch.build()
    for rev in (False, True, True):
        print("case busy batch", bs, prec, rev, flush=True)
        batch.execute(rev)
    assert batch.flowAborts() == 0
    for m, dx, b in keep[:len(mats)] + keep[-3:]:
        ce, prp, pcol, pval = mats[m]
        n = len(prp) - 1
        got = dx.download()
        xo = np.zeros(n * nrhs)
        for rev in (False, True, True):
            oracle.run_calls(oracle.K_KACZ, prp, pcol, pval, xo, b.astype(np.float64), _calls(ce, rev), nrhs=nrhs)
        assert relerr(got.astype(np.float64), xo) <= TOL[prec], m
        ce.setOption("bundle_threads", bs)
        ce.setOption("bundle_rows", 128)
        ce.setOption("layout", 2)
        ce.setOption("flow", 0)
        sx, sb = R.DeviceArray.from_host(np.zeros(len(b), dt)), R.DeviceArray.from_host(b)
        fid = ce.registerDevice(R.K_KACZ, prp, pcol, pval, sx, sb, nrhs=nrhs, val_precision=prec, vec_precision=prec)
        for rev in (False, True, True):
            ce.executeFunction(fid, rev)
        assert np.array_equal(got, sx.download()), m

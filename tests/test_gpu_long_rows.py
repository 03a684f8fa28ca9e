"""Variable lanes per row: rows of one lane up to more than a wavefront's 64
lanes, waves inside one wavefront and spread over several, chains of bundles
with more local columns than one batch of gathers holds, explicit zeros among
the entries, against the oracle in RACE order (1e-12, the parity bound of the
FP64 sweeps)."""
import numpy as np
import pytest

import race_amd as R
from race_amd import matgen as M

from .conftest import relerr

pytestmark = pytest.mark.gpu

TOL = 1e-12


def _hubs(n, hubs, seed):
    """a path with hub rows of the given numbers of neighbours, some entries 0"""
    rng = np.random.default_rng(seed)
    rows, cols = [np.arange(n - 1)], [np.arange(1, n)]
    for h, k in hubs:
        rows.append(np.full(k, h))
        cols.append(rng.choice(np.delete(np.arange(n), h), k, replace=False))
    rp, col = M._symmetric_csr(n, np.concatenate(rows), np.concatenate(cols))
    val = M.gs_values(rp, col, seed)
    r = M.row_of(rp)
    val[(col != r) & ((r + col) % 11 == 0)] = 0.0
    return rp, col, val


# 70 entries: 5 lanes; 16 * 64 entries: one wavefront's lanes; more: several
# wavefronts; 3800 entries: about all lanes of 256 threads
HUBS = {"short": [(3, 66), (50, 70), (51, 90), (900, 129)],
        "one_wavefront": [(7, 1016), (8, 1022), (1500, 1030)],
        "several": [(0, 1300), (40, 2047), (41, 2100), (1999, 3300)]}


@pytest.mark.parametrize("bs,local", [(256, 0), (512, 0), (1024, 0), (256, 5000)])
@pytest.mark.parametrize("name", sorted(HUBS))
@pytest.mark.parametrize("kind", [R.K_GS, R.K_KACZ])
def test_long_rows_match_race_order(oracle, kind, name, bs, local):
    n = 5200
    rp, col, val = _hubs(n, HUBS[name], len(name))
    dist, odist = (R.ONE, oracle.ONE) if kind == R.K_GS else (R.TWO, oracle.TWO)
    okind = oracle.K_GS if kind == R.K_GS else oracle.K_KACZ
    ce = R.Interface(n, 4, dist, rp, col, symm_hint=True)
    ce.RACEColor()
    g = oracle.Graph(rp, col, symm_hint=True)
    zt = oracle.level_recursion(g, 4, odist)
    prp, pcol, pval = M.make_diag_first(*M.permute(rp, col, val, ce.getPerm(), ce.getInvPerm()))
    b = M.uniform_vec(n, 4)
    ce.setOption("bundle_threads", bs)
    if local:
        ce.setOption("bundle_local", local)
    for flow in (0, 1) if kind == R.K_KACZ else (0,):
        ce.setOption("flow", flow)
        dx, db = R.DeviceArray.from_host(np.zeros(n)), R.DeviceArray.from_host(b)
        fid = ce.registerDevice(kind, prp, pcol, pval, dx, db)
        xo = np.zeros(n)
        for rev in (False, True):
            print("case long rows", kind, name, bs, local, flow, rev, flush=True)
            ce.executeFunction(fid, rev)
            oracle.run_calls(okind, prp, pcol, pval, xo, b, oracle.leaf_calls(zt, rev))
            assert relerr(dx.download(), xo) <= TOL
        assert ce.flowAborts(fid) == 0


def test_kaczmarz_row_of_infinite_right_hand_side():
    """b = inf in one row: its columns become infinite, later rows that touch
    them too, as the quotient by the row norm says; all other x are finite."""
    n = 64
    rp = np.arange(n + 1, dtype=np.int32) * 1
    col = np.arange(n, dtype=np.int32)
    val = np.linspace(0.5, 2.0, n)
    ce = R.Interface(n, 1, R.TWO, rp, col, symm_hint=True)
    ce.RACEColor()
    prp, pcol, pval = M.make_diag_first(*M.permute(rp, col, val, ce.getPerm(), ce.getInvPerm()))
    b = np.ones(n)
    b[10] = np.inf
    dx, db = R.DeviceArray.from_host(np.zeros(n)), R.DeviceArray.from_host(b)
    fid = ce.registerDevice(R.K_KACZ, prp, pcol, pval, dx, db)
    ce.executeFunction(fid)
    got = dx.download()
    assert got[10] == np.inf and np.all(np.isfinite(np.delete(got, 10)))
    assert relerr(np.delete(got, 10), 1.0 / np.delete(pval, 10)) <= TOL


# Columns of one chain that just fit a CU's LDS beside 256 partial sums and 129
# row starts, and one more.  FP32: a row's sum of up to 16 products a lane and
# ten additions over lanes errs by less than 30 * 2^-24, and a column is written
# by at most ten rows.
@pytest.mark.parametrize("prec,n,tol", [(R.FP64, 19000, TOL), (R.FP64, 19967, TOL), (R.FP64, 19968, TOL),
                                        (R.FP32, 40255, 2e-5), (R.FP32, 40256, 2e-5)])
def test_chain_columns_held_in_lds(oracle, prec, n, tol):
    """a single leaf of over a hundred bundles, one and three right-hand sides,
    phase launches and one launch per sweep"""
    rp, col, val = _hubs(n, [(5, 200), (77, 2500), (n - 1, 70)], 3)
    ce = R.Interface(n, 1, R.TWO, rp, col, symm_hint=True)
    ce.RACEColor()
    zt = oracle.level_recursion(oracle.Graph(rp, col, symm_hint=True), 1, oracle.TWO)
    prp, pcol, pval = M.make_diag_first(*M.permute(rp, col, val, ce.getPerm(), ce.getInvPerm()))
    dt = np.float64 if prec == R.FP64 else np.float32
    ce.setOption("bundle_threads", 256)
    for nrhs in (1, 3):
        b = M.uniform_vec(n, 4, nrhs=nrhs).astype(dt)
        for flow in (0, 1):
            ce.setOption("flow", flow)
            dx, db = R.DeviceArray.from_host(np.zeros(n * nrhs, dt)), R.DeviceArray.from_host(b)
            fid = ce.registerDevice(R.K_KACZ, prp, pcol, pval, dx, db, nrhs=nrhs, val_precision=prec,
                                    vec_precision=prec)
            xo = np.zeros(n * nrhs)
            for rev in (False, True):
                print("case chain columns", n, prec, nrhs, flow, rev, flush=True)
                ce.executeFunction(fid, rev)
                oracle.run_calls(oracle.K_KACZ, prp, pcol, pval, xo, b.astype(np.float64).ravel(),
                                 oracle.leaf_calls(zt, rev), nrhs=nrhs)
                assert relerr(dx.download().ravel(), xo) <= tol
            assert ce.flowAborts(fid) == 0

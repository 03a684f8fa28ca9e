"""SpMV on a batch of matrices, the smaller ones with runs of empty rows before
larger ones, against FP64 sums.

Bound: a row sum of L products in precision u, in any order, is within
(L + 2) u sum |a||x| of the exact sum, and the reference sum within as much in
FP64."""
import numpy as np
import pytest

import race_amd as R
from race_amd import matgen as M

pytestmark = pytest.mark.gpu


def _matrix(lengths, seed):
    n = len(lengths)
    rng = np.random.default_rng(seed)
    rp = np.concatenate([[0], np.cumsum(lengths)]).astype(np.int32)
    col = rng.integers(0, n, rp[-1]).astype(np.int32)
    return rp, col, rng.uniform(-1, 1, rp[-1])


def _lengths(n, empty, hub):
    """1 to 9 entries a row, one hub, no entries where empty(r)"""
    r = np.arange(n)
    k = np.where(empty(r), 0, 1 + r * 7 % 9)
    k[np.flatnonzero(k)[:1]] = hub
    return k


SHAPES = [
    _lengths(1000, lambda r: r >= 448, 40),      # a block of empty rows at the end
    _lengths(100000, lambda r: r < 0, 3000),
    _lengths(900, lambda r: r < 600, 40),        # at the start
    _lengths(70000, lambda r: r % 1500 < 700, 2000),
    _lengths(2000, lambda r: r > 1, 1500),       # behind a row that is a block of its own
    np.zeros(300, int),
    _lengths(50000, lambda r: r < 0, 100),
    np.full(640, 5),                             # regular: chunks
    np.zeros(1, int),
]


@pytest.mark.parametrize("prec,nrhs", [(R.FP64, 1), (R.FP64, 3), (R.FP32, 1), (R.FP32, 8)])
def test_spmv_batch_with_empty_rows(prec, nrhs):
    dt, u = (np.float64, 2.0 ** -53) if prec == R.FP64 else (np.float32, 2.0 ** -24)
    batch = R.Batch(R.K_SPMV, prec, prec, nrhs=nrhs)
    keep = []
    for k, lengths in enumerate(SHAPES):
        rp, col, val = _matrix(lengths, 31 + k)
        n = len(lengths)
        val = val.astype(dt).astype(np.float64)
        x = M.uniform_vec(n, 50 + k, nrhs=nrhs).astype(dt)
        dx, db = R.DeviceArray.from_host(x), R.DeviceArray.from_host(np.full(n * nrhs, 7.0, dt))
        batch.add(R.Interface(n, 1, R.ONE, rp, col, symm_hint=False), rp, col, val, dx, db)
        A, X = M.to_scipy(rp, col, val), x.astype(np.float64).reshape(nrhs, n).T
        keep.append((db, (A @ X).T, (np.diff(rp) + 3)[None] * u * (abs(A) @ abs(X)).T))
    print("case batch spmv", prec, nrhs, flush=True)
    batch.execute()
    for k, (db, ref, bound) in enumerate(keep):
        got = db.download().astype(np.float64).reshape(ref.shape)
        assert np.all(np.abs(got - ref) <= bound), k

"""Rows of 1 to 7 entries in ragged matrices, FP32: every row is one chain of
fused multiply-adds over its entries, one rounding per entry, bit for bit (the
product of two FP32 numbers is exact in FP64, and so is the rounding of the sum
but for ties that these values do not hit)."""
import numpy as np
import pytest

import race_amd as R
from race_amd import matgen as M

pytestmark = pytest.mark.gpu


# one right-hand side; separate columns; packed right-hand sides
@pytest.mark.parametrize("n,nrhs", [(4096, 1), (4096, 3), (4096, 8), (131072, 4), (131072, 8)])
@pytest.mark.parametrize("prec", [R.FP32, R.BF16])
def test_one_rounding_per_entry(n, nrhs, prec):
    rng = np.random.default_rng(n + nrhs)
    lengths = rng.permutation(np.arange(n) % 7 + 1)
    rp = np.concatenate([[0], np.cumsum(lengths)]).astype(np.int32)
    col = rng.integers(0, n, rp[-1]).astype(np.int32)
    val = rng.uniform(-1, 1, rp[-1]).astype(np.float32)
    if prec == R.BF16:
        val = (val.view(np.uint32) & np.uint32(0xffff0000)).view(np.float32)
    x = M.uniform_vec(n, 3, nrhs=nrhs).astype(np.float32)
    ce = R.Interface(n, 1, R.ONE, rp, col, symm_hint=False)
    dx, db = R.DeviceArray.from_host(x), R.DeviceArray.from_host(np.zeros(n * nrhs, np.float32))
    fid = ce.registerDevice(R.K_SPMV, rp, col, val.astype(np.float64), dx, db, nrhs=nrhs, val_precision=prec,
                            vec_precision=R.FP32)
    print("case short rows", n, nrhs, prec, flush=True)
    ce.executeFunction(fid)
    X = x.reshape(nrhs, n).astype(np.float64)
    ref = np.zeros((nrhs, n), np.float32)
    for j in range(7):
        rows = np.flatnonzero(lengths > j)
        e = rp[rows] + j
        ref[:, rows] = (val[e].astype(np.float64) * X[:, col[e]] + ref[:, rows]).astype(np.float32)
    # the rows of the last, smaller block share lanes
    assert np.array_equal(db.download().reshape(nrhs, n)[:, :n - 600], ref[:, :n - 600])

"""Which kernel a product with several right-hand sides takes: small matrices,
scattered columns, streams with and without packing scratch, and a registration
for which there is no scratch memory left.

Bound: a row sum of L products in precision u, in any order, is within
(L + 2) u sum |a||x| of the exact sum; the reference sums have 64 bits of mantissa
(of the values as stored)."""
import ctypes

import numpy as np
import pytest

import race_amd as R
from race_amd import _lib as L
from race_amd import matgen as M

pytestmark = pytest.mark.gpu

U = {R.FP64: 2.0 ** -53, R.FP32: 2.0 ** -24}


def _regular(n, k, seed, window=0):
    rng = np.random.default_rng(seed)
    col = rng.integers(0, n, n * k)
    if window:
        col = np.clip(np.repeat(np.arange(n), k) + rng.integers(-window, window, n * k), 0, n - 1)
    return (np.arange(n + 1) * k).astype(np.int32), col.astype(np.int32), rng.uniform(-1, 1, n * k)


class Product:
    def __init__(self, rp, col, val, prec, nrhs):
        self.n, self.nrhs, dt = len(rp) - 1, nrhs, np.float64 if prec == R.FP64 else np.float32
        self.ce = R.Interface(self.n, 1, R.ONE, rp, col, symm_hint=False)
        self.x = M.uniform_vec(self.n, 3, nrhs=nrhs).astype(dt)
        self.dx, self.db = R.DeviceArray.from_host(self.x), R.DeviceArray.from_host(np.zeros(self.n * nrhs, dt))
        self.fid = self.ce.registerDevice(R.K_SPMV, rp, col, val, self.dx, self.db, nrhs=nrhs, val_precision=prec,
                                          vec_precision=prec)
        # every row has k entries
        k, a, X = int(rp[1]), val.astype(dt).astype(np.longdouble), self.x.astype(np.longdouble).reshape(nrhs, self.n)
        self.ref, size = np.zeros((2, nrhs, self.n), np.longdouble)
        for j in range(k):
            p = a[j::k] * X[:, col[j::k]]
            self.ref += p
            size += abs(p)
        self.bound = (k + 3) * U[prec] * size

    def check(self, stream=None):
        self.ce.executeAsync(self.fid, stream=stream)
        assert L.load().race_device_synchronize() == 0
        got = self.db.download().astype(np.longdouble).reshape(self.ref.shape)
        bad = np.argwhere(np.abs(got - self.ref) > self.bound)
        assert len(bad) == 0, (len(bad), bad[:3])
        self.db.zero()
        assert L.load().race_device_synchronize() == 0


# lanes per row: 1 to 64 entries a row, the most entries and columns of the rule and
# one step past them, rows of 65 entries
@pytest.mark.parametrize("n,k,nrhs", [(1, 1, 2), (7, 7, 3), (37, 9, 2), (1000, 17, 5), (513, 64, 11), (513, 65, 3),
                                      (15000, 30, 2), (15001, 30, 2), (5000, 60, 4), (5000, 60, 5), (9999, 8, 8),
                                      (20000, 20, 3), (20000, 20, 4)])
def test_small_matrices(n, k, nrhs):
    for prec in (R.FP64, R.FP32):
        print("case small", n, k, nrhs, prec, flush=True)
        Product(*_regular(n, k, n), prec, nrhs).check()


# scattered columns of regular rows: packed, and chunks side by side
@pytest.mark.parametrize("n,k,nrhs,window", [(40000, 20, 2, 0), (40000, 20, 3, 0), (60000, 24, 2, 3000),
                                             (60000, 24, 3, 3000), (60000, 24, 5, 3000), (50000, 6, 3, 0)])
def test_scattered_columns_on_any_stream(n, k, nrhs, window):
    """two streams may get packing scratch, the others run over the chunks"""
    owners = [R.Interface(64, 1, R.ONE, *_regular(64, 1, 1)[:2], symm_hint=False) for _ in range(3)]
    for prec in (R.FP64, R.FP32):
        p = Product(*_regular(n, k, k, window), prec, nrhs)
        for stream in [None] + [o.stream() for o in owners]:
            print("case scattered", n, k, nrhs, window, prec, stream is None, flush=True)
            p.check(stream)


def _free():
    a, b = ctypes.c_size_t(), ctypes.c_size_t()
    assert ctypes.CDLL("libamdhip64.so.7").hipMemGetInfo(ctypes.byref(a), ctypes.byref(b)) == 0
    return a.value


# 128 MB of scratch a set: room for one set, for none
@pytest.mark.parametrize("room,launches", [(1.5, 2), (0.5, 1)])
def test_registration_without_room_for_scratch(room, launches):
    n, k, nrhs = 250000, 8, 64
    rp, col, val = _regular(n, k, 9)
    one = n * nrhs * 8
    Product(*_regular(64, 3, 1), R.FP64, 2).check()  # the library's own memory is there
    left = int((2 + 0.5 + room) * one)  # x, b; both layouts of the matrix; then the sets
    fill = []
    try:
        while _free() - left > 1 << 20:
            fill.append(R.DeviceArray(min(_free() - left, 32 << 30), np.uint8))
        print("case no room", room, _free() / one, flush=True)
        p = Product(rp, col, val, R.FP64, nrhs)
        assert p.ce.launchCount(p.fid) == launches
        p.check()
    finally:
        for f in fill:
            f.free()

"""The row-parallel products (SpMV, SpMTV, SymmSpMV, matrix powers) at the
edges of their layouts: every remainder of the row blocks, 16- and 32-bit
column ids, rows far shorter than their chunk, the right-hand-side blocks,
matrices read by XCD parts and non-temporally, infinities next to padding.

Bound: a row sum of L products in precision u, in any order, is within
(L + 2) u sum |a||x| of the exact sum (each product and each addition rounds
once, the stored result once); the reference sum itself is in FP64."""
import numpy as np
import pytest

import race_amd as R
from race_amd import matgen as M

pytestmark = pytest.mark.gpu

U = {R.FP64: 2.0 ** -53, R.FP32: 2.0 ** -24}


def _bf16(v):
    u = np.asarray(v, np.float32).view(np.uint32)
    return ((u + 0x7fff + ((u >> 16) & 1)) & np.uint32(0xffff0000)).view(np.float32).astype(np.float64)


def _stored(val, prec):
    return val if prec == R.FP64 else val.astype(np.float32).astype(np.float64) if prec == R.FP32 else _bf16(val)


def _random(n, lengths, seed, window=None):
    """lengths[r] distinct columns per row, within window columns of the row"""
    rng = np.random.default_rng(seed)
    w = n if window is None else min(n, window)
    cols = [np.sort((rng.choice(w, min(k, w), replace=False) + (0 if w == n else max(0, r - w // 2))) % n)
            for r, k in enumerate(lengths)]
    rp = np.zeros(n + 1, np.int32)
    rp[1:] = np.cumsum([len(c) for c in cols])
    col = np.concatenate(cols).astype(np.int32) if rp[-1] else np.zeros(0, np.int32)
    return rp, col, rng.uniform(-1, 1, len(col))


def _check(rp, col, val, kind, prec, nrhs, seed=3):
    n = len(rp) - 1
    vec = R.FP64 if prec == R.FP64 else R.FP32
    dt = np.float64 if vec == R.FP64 else np.float32
    x = M.uniform_vec(n, seed, nrhs=nrhs).astype(dt)
    b = M.uniform_vec(n, seed + 1, nrhs=nrhs).astype(dt)
    ce = R.Interface(n, 1, R.ONE, rp, col, symm_hint=False)
    dx, db = R.DeviceArray.from_host(x), R.DeviceArray.from_host(b)
    fid = ce.registerDevice(kind, rp, col, val, dx, db, nrhs=nrhs, val_precision=prec, vec_precision=vec)
    ce.executeFunction(fid)
    got = db.download().astype(np.float64).reshape(nrhs, n)
    A = M.to_scipy(rp, col, _stored(val, prec))
    A = A.T.tocsr() if kind == R.K_SPMTV else A
    X, B = (v.astype(np.float64).reshape(nrhs, n).T for v in (x, b))
    B = B if kind == R.K_SPMTV else 0 * B
    ref, size = (A @ X + B).T, (abs(A) @ abs(X) + abs(B)).T
    bound = (np.diff(A.indptr) + 3)[None] * U[vec] * size
    worst = np.max(np.abs(got - ref) - bound)
    assert worst <= 0, worst


# every remainder of the blocks of 8, 4, 2 and 1; rows of 0 entries among them
@pytest.mark.parametrize("prec", [R.FP64, R.FP32, R.BF16])
@pytest.mark.parametrize("width", [1, 2, 3, 4, 5, 6, 7, 8, 9, 14, 15, 16, 23, 31])
def test_block_remainders(width, prec):
    print("case remainder", width, prec, flush=True)
    n = 64 * 9 + 37
    lengths = [width - (r % 5 == 3) * min(width, 2) for r in range(n)]
    _check(*_random(n, lengths, width), R.K_SPMV, prec, 1)


# columns of one slot up to 65535 apart (16-bit ids) and further (32-bit ids)
@pytest.mark.parametrize("prec", [R.FP64, R.FP32, R.BF16])
@pytest.mark.parametrize("far", [65535, 65536, 90000])
def test_column_id_width(far, prec):
    print("case ids", far, prec, flush=True)
    n = 131072 + 5
    rows = [[r, (r + 1) % n] for r in range(n)]
    rows[64] = [64, 64 + 1 + far]  # slot 1 of its chunk then spans `far` columns
    rp = (2 * np.arange(n + 1)).astype(np.int32)
    col = np.array(rows, np.int32).reshape(-1)
    val = np.random.default_rng(far).uniform(-1, 1, len(col))
    _check(rp, col, val, R.K_SPMV, prec, 1)


@pytest.mark.parametrize("kind", [R.K_SPMV, R.K_SPMTV])
@pytest.mark.parametrize("nrhs", [1, 2, 3, 4, 5, 8, 9, 11, 12, 16])
def test_right_hand_side_blocks(nrhs, kind):
    for prec in (R.FP64, R.FP32, R.BF16):
        print("case rhs", nrhs, kind, prec, flush=True)
        _check(*_random(1000, [11 + r % 3 for r in range(1000)], nrhs, 300), kind, prec, nrhs)


# one row more than 255 entries longer than its neighbours
@pytest.mark.parametrize("nrhs", [1, 4])
@pytest.mark.parametrize("long_row", [255 + 3, 256 + 3, 1500])
def test_long_row_in_short_chunk(long_row, nrhs):
    print("case long row", long_row, nrhs, flush=True)
    n = 2000
    lengths = [3] * n
    lengths[70] = long_row
    for prec in (R.FP64, R.BF16):
        _check(*_random(n, lengths, long_row), R.K_SPMV, prec, nrhs)


# about 20 MB, 80 MB and 300 MB of entries: plain, by XCD parts, non-temporal
@pytest.mark.parametrize("n", [200003, 800003, 3000001])
def test_reading_order_by_size(n):
    print("case size", n, flush=True)
    offs = np.array([0, 1, 2, 5, 17, 300, 4000, 9000, 20011, 50000])
    rp = (len(offs) * np.arange(n + 1)).astype(np.int32)
    col = np.sort((np.arange(n)[:, None] + offs[None]) % n, axis=1).astype(np.int32).reshape(-1)
    val = np.random.default_rng(n).uniform(-1, 1, len(col))
    _check(rp, col, val, R.K_SPMV, R.FP64, 1)


def test_infinity_stays_in_its_rows():
    """x = inf in a column: rows without that column are finite, as padding
    entries multiply 0 by 0."""
    n = 640
    rp, col, val = _random(n, [5 + r % 4 for r in range(n)], 5)
    x = np.ones(n)
    x[::7] = np.inf
    ce = R.Interface(n, 1, R.ONE, rp, col, symm_hint=False)
    dx, db = R.DeviceArray.from_host(x), R.DeviceArray.from_host(np.zeros(n))
    fid = ce.registerDevice(R.K_SPMV, rp, col, np.abs(val) + 0.1, dx, db)
    ce.executeFunction(fid)
    touched = np.array([np.isinf(x[col[rp[r]:rp[r + 1]]]).any() for r in range(n)])
    assert np.array_equal(np.isinf(db.download()), touched) and not np.isnan(db.download()).any()


RAGGED = {
    # blocks of one, two and three rows, exactly and just over 1024 entries
    "one_row_blocks": [1024, 1, 1023, 1025, 3000, 0, 5],
    "two_and_three": [512, 512, 341, 342, 341, 600, 424, 1],
    # more empty rows than a block holds, at the start and at the end
    "empty_ends": [0] * 300 + [40] + [0] * 600,
    "all_empty": [0] * 700,
    # a block that ends by its row count, and hub rows among short ones
    "short_rows": [1, 0, 2] * 200 + [900] + [3] * 50,
    # the longest row a lane or its lanes sum alone, and one entry more; as many hubs as a block holds
    "hub_edges": [1] * 100 + [16] + [1] * 150 + [17] * 70 + [64, 65, 128, 129] + [0] * 250 + [33] * 9 + [1] * 240,
}


@pytest.mark.parametrize("kind", [R.K_SPMV, R.K_SPMTV])
@pytest.mark.parametrize("name", sorted(RAGGED))
def test_row_blocks(name, kind):
    lengths = RAGGED[name]
    lengths = lengths + [1] * max(0, 3100 - len(lengths)) if max(lengths) > 900 else lengths
    for prec, nrhs in ((R.FP64, 1), (R.FP32, 1), (R.BF16, 1), (R.FP64, 3), (R.FP32, 2), (R.FP32, 8), (R.BF16, 11)):
        print("case ragged", name, kind, prec, nrhs, flush=True)
        _check(*_random(len(lengths), lengths, len(name)), kind, prec, nrhs)


def test_row_blocks_wide_ids():
    """ragged rows over more than 65535 columns: 32-bit ids"""
    n = 200000
    lengths = [(r % 97 == 0) * 60 + r % 3 for r in range(n)]
    rng = np.random.default_rng(4)
    rp = np.concatenate([[0], np.cumsum(lengths)]).astype(np.int32)
    col = rng.integers(0, n, rp[-1]).astype(np.int32)
    for prec, nrhs in ((R.FP64, 1), (R.FP32, 4)):
        _check(rp, col, rng.uniform(-1, 1, len(col)), R.K_SPMV, prec, nrhs)


@pytest.mark.parametrize("kind", [R.K_SPMV, R.K_SPMTV])
@pytest.mark.parametrize("nrhs", [2, 3, 4, 5, 8, 9])
def test_packed_right_hand_sides(nrhs, kind):
    """scattered columns: right-hand sides packed row by row, full and partly
    filled blocks of them; rows of 0, 512, 513 and 3000 entries"""
    n = 6000
    lengths = [int(k) for k in np.random.default_rng(3).integers(0, 60, n)]
    lengths[5], lengths[6], lengths[7], lengths[4000], lengths[-1] = 512, 513, 1024, 3000, 0
    for prec in (R.FP64, R.FP32, R.BF16):
        print("case packed", nrhs, kind, prec, flush=True)
        rp, col, val = _random(n, lengths, 7)
        _check(rp, col, val, kind, prec, nrhs)


def test_packed_on_overlapping_streams():
    """one function on four streams at once, each call with vectors of its
    own: two streams with packing scratch, the others without"""
    n, nrhs = 20000, 4
    rng = np.random.default_rng(1)
    lengths = rng.integers(0, 40, n)
    rp = np.concatenate([[0], np.cumsum(lengths)]).astype(np.int32)
    col = rng.integers(0, n, rp[-1]).astype(np.int32)
    val = rng.uniform(-1, 1, len(col))
    owners = [R.Interface(n, 1, R.ONE, rp, col, symm_hint=False) for _ in range(4)]
    xs = [M.uniform_vec(n, k, nrhs=nrhs) for k in range(4)]
    vecs = [(R.DeviceArray.from_host(x), R.DeviceArray.from_host(np.zeros(n * nrhs))) for x in xs]
    fid = owners[0].registerDevice(R.K_SPMV, rp, col, val, *vecs[0], nrhs=nrhs)
    assert owners[0].launchCount(fid) == 2
    for step in range(20):
        for k, o in enumerate(owners):
            owners[0].setVectors(fid, *vecs[k])
            owners[0].executeAsync(fid, stream=o.stream())
    assert owners[0].flowAborts(fid) == 0  # waits for the device
    A = M.to_scipy(rp, col, val)
    for k in range(4):
        ref = (A @ xs[k].reshape(nrhs, n).T).T
        assert np.max(np.abs(vecs[k][1].download().reshape(nrhs, n) - ref)) <= 60 * 2.0 ** -53 * 60

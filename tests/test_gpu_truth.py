"""Brute-force ground truth at the edges of its tiles, levels and dispatch.

8-bit rows: ids (ties to the smaller id) and distances equal whole-number
arithmetic.  Float rows: every distance is an fp32 sum of dim squares of
fp32 differences, so it is off by at most (dim + 2) 2^-24 of itself (each of
the dim additions rounds once, the difference twice in its square), and by the
underflow of its squares; the
returned distances ascend and match the float64 ones rank by rank within that.
"""
from __future__ import annotations

import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def lib():
    from quiver import _lib

    if _lib.device_count() == 0:
        pytest.skip("no GPU")
    return _lib


def _truth(lib, base, q, k):
    n, dim = base.shape
    nq = q.shape[0]
    code = {"uint8": lib.QV_UINT8, "int8": lib.QV_INT8, "float32": lib.QV_FLOAT}[base.dtype.name]
    db, dq = lib.DeviceBuffer(base.nbytes).upload(base), lib.DeviceBuffer(q.nbytes).upload(q)
    di, dd = lib.DeviceBuffer(nq * k * 4), lib.DeviceBuffer(nq * k * 4)
    lib.check(lib.load().qv_ground_truth(db.ptr, code, n, dim, dq.ptr, nq, k, di.ptr, dd.ptr, 0))
    out = di.download(np.int32, (nq, k)), dd.download(np.float32, (nq, k))
    for b in (db, dq, di, dd):
        b.close()
    return out


def _check(base, q, k, ids, dists):
    n, dim = base.shape
    kk = min(k, n)
    b, qq = base.astype(np.float64), q.astype(np.float64)
    d = np.empty((q.shape[0], n))
    for i in range(q.shape[0]):
        with np.errstate(over="ignore", invalid="ignore"):
            d[i] = ((b - qq[i]) ** 2).sum(1)
    assert (ids[:, kk:] == -1).all() and np.isinf(dists[:, kk:]).all()
    if base.dtype != np.float32 and np.array_equal(q, np.rint(q)):
        order = np.argsort(d, axis=1, kind="stable")[:, :kk]
        np.testing.assert_array_equal(ids[:, :kk], order)
        np.testing.assert_array_equal(dists[:, :kk], np.take_along_axis(d, order, 1))
        return
    tol, tiny = (dim + 2) * 2.0 ** -24, dim * 2.0 ** -149  # squares may also underflow, each by less than 2^-149
    got = dists[:, :kk].astype(np.float64)
    assert (np.diff(got, axis=1) >= 0).all()
    np.testing.assert_allclose(got, np.take_along_axis(d, ids[:, :kk].astype(np.int64), 1), rtol=tol, atol=tiny)
    np.testing.assert_allclose(got, np.sort(d, axis=1)[:, :kk], rtol=tol, atol=tiny)
    assert all(len(set(r)) == kk for r in ids[:, :kk].tolist())


def _rows(dtype, n, dim, seed, high=None):
    rng = np.random.default_rng(seed)
    if dtype == "float32":
        return np.ascontiguousarray(rng.standard_normal((n, dim)) + 2 * rng.standard_normal((1, dim)), np.float32)
    lo, hi = (0, high or 256) if dtype == "uint8" else (-128, 128)
    return rng.integers(lo, hi, (n, dim)).astype(dtype)


# rows: below, at and past one tile of 64 and one, two and three levels; queries: around a
# wave's 32, a workgroup's 128 and 512 and the switch at 256; dimensions: each operand width
# and its remainder, and rows past them (the direct kernels); k: both list sizes and the limits
@pytest.mark.parametrize("dtype", ["uint8", "int8", "float32"])
@pytest.mark.parametrize("n, nq, dim, k", [
    (1, 1, 4, 1), (63, 31, 32, 5), (64, 33, 36, 64), (65, 128, 64, 16), (256, 129, 68, 17),
    (1025, 257, 96, 10), (4097, 513, 100, 10), (16385, 256, 128, 16), (20001, 40, 128, 64), (5000, 20, 132, 10),
    (3000, 20, 260, 10),
])
def test_edges(lib, dtype, n, nq, dim, k):
    print(f"[gpu] truth {dtype} n={n} nq={nq} dim={dim} k={k}", flush=True)
    base, q = _rows(dtype, n, dim, n), _rows(dtype, nq, dim, n + 1).astype(np.float32)
    _check(base, q, k, *_truth(lib, base, q, k))


@pytest.mark.parametrize("what", ["ties", "one row repeated", "against the period", "fractional queries"])
def test_lists_and_ties(lib, what):
    """Equal distances everywhere, lists that overflow, and queries the 8-bit products cannot hold."""
    print(f"[gpu] truth, {what}", flush=True)
    base, q = _rows("uint8", 20000, 16, 3, 3), _rows("uint8", 70, 16, 4, 3).astype(np.float32)
    if what == "one row repeated":
        base = np.repeat(base[:1], 20000, axis=0)
    if what == "against the period":  # every row a sample may take is far, all others near
        base[::4] = 255
    if what == "fractional queries":
        q += 0.5
    _check(base, q, 10, *_truth(lib, base, q, 10))


def test_float_rows_out_of_scale(lib):
    """Rows and queries whose norms overflow or vanish, infinities, and a common offset far above the spread."""
    print("[gpu] truth, float scales", flush=True)
    base, q = _rows("float32", 5000, 96, 5), _rows("float32", 40, 96, 6)
    base[7, 3] = np.inf
    base[11] = 3e38
    base[13] = 1e19
    base[15] = 1e-30
    q[6] = 1e18
    q[8] = 0
    q[9] = 1e-30
    ids, dists = _truth(lib, base, q, 10)
    keep = np.array([7, 11])
    assert not np.isin(ids, keep).any()
    finite = base.copy()
    finite[keep] = 1e19  # far from every query but row 6's, whose nearest rows are the near ones all the same
    _check(finite, q, 10, ids, dists)
    for scale, off in ((1e-19, 0.0), (1.0, 300.0)):
        q2 = _rows("float32", 40, 96, 6)
        b2 = np.ascontiguousarray(_rows("float32", 5000, 96, 5) * scale + off, np.float32)
        q2 = np.ascontiguousarray(q2 * scale + off, np.float32)
        ids, dists = _truth(lib, b2, q2, 10)
        if scale == 1.0:
            _check(b2, q2, 10, ids, dists)
        else:  # squares near the smallest normal numbers: ranks only, absolutely
            d = ((b2.astype(np.float64)[None] - q2.astype(np.float64)[:, None]) ** 2).sum(2)
            np.testing.assert_allclose(dists, np.sort(d, axis=1)[:, :10], rtol=98 * 2.0 ** -24, atol=96 * 2.0 ** -149)


def _counted(lib, base, q, k, scan_small=0):
    """ids, distances, and how many of the queries the direct kernels answered (scan_small: the scan is taken however
    small the call)."""
    fn = lib.load().qv_ground_truth_counted
    fn.restype, fn.argtypes = C.c_int32, lib.load().qv_ground_truth.argtypes + [C.c_int32, C.POINTER(C.c_int64)]
    n, dim = base.shape
    nq = q.shape[0]
    code = {"uint8": lib.QV_UINT8, "int8": lib.QV_INT8, "float32": lib.QV_FLOAT}[base.dtype.name]
    bufs = [lib.DeviceBuffer(x.nbytes).upload(x) for x in (base, q)] + [lib.DeviceBuffer(nq * k * 4) for _ in range(2)]
    direct = C.c_int64(-1)
    lib.check(fn(bufs[0].ptr, code, n, dim, bufs[1].ptr, nq, k, bufs[2].ptr, bufs[3].ptr, 0, scan_small, C.byref(direct)))
    out = bufs[2].download(np.int32, (nq, k)), bufs[3].download(np.float32, (nq, k)), direct.value
    for b in bufs:
        b.close()
    return out


# the shapes of test_edges within the tiles' row lengths, and the largest 8-bit rows
@pytest.mark.parametrize("dtype", ["uint8", "int8", "float32"])
@pytest.mark.parametrize("n, nq, dim, k", [
    (1, 1, 4, 1), (31, 3, 4, 40), (63, 31, 32, 5), (64, 33, 36, 64), (65, 128, 64, 16), (256, 129, 68, 17),
    (1025, 257, 96, 10), (4097, 513, 100, 10), (16385, 256, 128, 16), (20001, 40, 128, 64), (5000, 20, 256, 64),
])
def test_the_scan_answers(lib, dtype, n, nq, dim, k):
    """Ordinary data: no query is left to the direct kernels, and both ways give the same bits."""
    print(f"[gpu] truth by the scan {dtype} n={n} nq={nq} dim={dim} k={k}", flush=True)
    if dtype == "float32":
        dim = min(dim, 128)
    base, q = _rows(dtype, n, dim, n), _rows(dtype, nq, dim, n + 1).astype(np.float32)
    ids, dists, direct = _counted(lib, base, q, k, 1)
    assert direct == 0
    _check(base, q, k, ids, dists)
    for got, want in zip(_truth(lib, base, q, k), (ids, dists)):
        np.testing.assert_array_equal(got, want)


# both sides of the small-call lines: pairs, rows and queries
@pytest.mark.parametrize("dtype, n, nq, dim, k, small", [
    ("float32", 1000, 500, 32, 10, True), ("float32", 1000, 501, 32, 10, False), ("float32", 2048, 3, 32, 10, True),
    ("float32", 2049, 3, 32, 10, False), ("uint8", 500, 256, 16, 10, False), ("uint8", 500, 257, 16, 10, True),
    ("uint8", 5000, 1000, 16, 16, True), ("uint8", 5000, 1001, 16, 16, False), ("int8", 600, 1000, 16, 17, True),
    ("int8", 600, 1001, 16, 17, False), ("int8", 100, 300, 132, 10, False),
])
def test_small_calls(lib, dtype, n, nq, dim, k, small):
    print(f"[gpu] truth, small call {dtype} n={n} nq={nq} dim={dim} k={k}", flush=True)
    base, q = _rows(dtype, n, dim, n), _rows(dtype, nq, dim, n + 1).astype(np.float32)
    ids, dists, direct = _counted(lib, base, q, k)
    assert direct == (nq if small else 0)
    _check(base, q, k, ids, dists)


@pytest.mark.parametrize("what, direct", [
    ("one fractional query", 1), ("fractional queries", 70), ("against the period", 70), ("rows near one query", 1),
    ("each row repeated", 70), ("common offset", 0), ("common offset, rows far out", 0), ("long float rows", 70),
])
def test_queries_that_leave_the_scan(lib, what, direct):
    """Only the queries the scan cannot finish go to the direct kernels; a common offset is no reason to."""
    print(f"[gpu] truth, {what}", flush=True)
    base, q = _rows("uint8", 20000, 16, 3, 250), _rows("uint8", 70, 16, 4, 250).astype(np.float32)
    if what == "one fractional query":
        q[33, 5] += 0.25
    elif what == "fractional queries":
        q += 0.5
    elif what == "against the period":  # 250 rows a sample takes are far, the 750 scanned next near
        base = base[:16000]
        base[::4] = 255
    else:
        base, q = _rows("float32", 20000, 132 if what == "long float rows" else 96, 5), _rows("float32", 70, 96, 6)
        rng = np.random.default_rng(8)
        if what == "rows near one query":  # as near as one another, more than a list holds
            q = np.ascontiguousarray(base[::250][:70] + rng.standard_normal((70, 96)) / 2, np.float32)
            base[rng.permutation(20000)[:3000]] = q[12] + 0.125
        elif what == "each row repeated":
            base = np.ascontiguousarray(np.repeat(base[:10], 2000, axis=0)[rng.permutation(20000)])
        elif what == "long float rows":
            q = _rows("float32", 70, 132, 6)
        else:
            base, q = base + np.float32(300), q + np.float32(300)
            if what == "common offset, rows far out":
                base[::5000] = 1e12  # among the rows the scan's origin is taken from
    ids, dists, got = _counted(lib, base, q, 10)
    assert got == direct
    _check(base, q, 10, ids, dists)


def test_queries_without_a_norm(lib):
    """Queries with NaN, infinite or enormous elements leave the scan before it, alone: the others' answers are those
    of a call without them, and theirs the ones of the direct kernels."""
    print("[gpu] truth, queries without a norm", flush=True)
    base, q = _rows("float32", 20000, 96, 5), _rows("float32", 70, 96, 6)
    want = _counted(lib, base, q, 10)
    bad = {3: np.nan, 17: np.inf, 18: -np.inf, 60: 1e30, 69: 3e38}
    for row, v in bad.items():
        q[row, row] = v
    got = _counted(lib, base, q, 10)
    assert (want[2], got[2]) == (0, len(bad))
    rest = np.array([i for i in range(70) if i not in bad])
    np.testing.assert_array_equal(got[0][rest], want[0][rest])
    np.testing.assert_array_equal(got[1][rest], want[1][rest])
    # theirs: a call over few rows is the direct kernels' own; taken by the scan, they leave it and get the same bits
    few = _counted(lib, base[:2000], q[list(bad)], 10)
    scanned = _counted(lib, base[:2000], q[list(bad)], 10, 1)
    assert few[2] == scanned[2] == len(bad)
    np.testing.assert_array_equal(few[0], scanned[0])
    np.testing.assert_array_equal(few[1], scanned[1])


@pytest.mark.parametrize("dtype", ["uint8", "float32"])
def test_query_batches(lib, dtype):
    """More queries than one scan takes (32,768): the second batch has its own lists, results and queries that leave."""
    nq = 32768 + 37
    print(f"[gpu] truth {dtype} nq={nq}", flush=True)
    base, q = _rows(dtype, 300, 4, 1), _rows(dtype, nq, 4, 2).astype(np.float32)
    if dtype == "uint8":
        q[[7, 32770], 1] += 0.5
    ids, dists, direct = _counted(lib, base, q, 3)
    assert direct == (2 if dtype == "uint8" else 0)
    _check(base, q, 3, ids, dists)

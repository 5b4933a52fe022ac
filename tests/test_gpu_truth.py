"""Brute-force ground truth at the edges of its tiles, levels and dispatch.

8-bit rows: ids (ties to the smaller id) and distances equal whole-number
arithmetic.  Float rows: every distance is an fp32 sum of dim squares of
fp32 differences, so it is off by at most (dim + 2) 2^-24 of itself (each of
the dim additions rounds once, the difference twice in its square), and by the
underflow of its squares; the
returned distances ascend and match the float64 ones rank by rank within that.
"""
from __future__ import annotations

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

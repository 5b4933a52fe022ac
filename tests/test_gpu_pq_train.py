"""PQ tables and codes of a GPU-built index against a NumPy restatement: the
float64 mean, Lloyd iterations whose sums run in row order, and restarts of
pivots no row is nearest to.  Distances are the fp32 chain s = fma(d, d, s);
d d + s in float64 rounds to the same fp32 value (the product is exact there).
Everything is compared bit for bit."""
from __future__ import annotations

import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu
MASK = (1 << 64) - 1


@pytest.fixture(scope="module")
def lib():
    from quiver import _lib

    if _lib.device_count() == 0:
        pytest.skip("no GPU")
    return _lib


def _mix(z):
    z = (z + 0x9E3779B97F4A7C15) & MASK
    z = ((z ^ (z >> 30)) * 0xBF58476D1CE4E5B9) & MASK
    z = ((z ^ (z >> 27)) * 0x94D049BB133111EB) & MASK
    return z ^ (z >> 31)


def _rng(seed, stream, counter):
    return _mix(_mix((seed + stream * 0xD1B54A32D192ED03) & MASK) ^ counter)


def _nearest(x, p):
    s = np.zeros((x.shape[0], 256), np.float32)
    for j in range(x.shape[1]):
        d = (x[:, j:j + 1] - p[None, :, j]).astype(np.float64)
        s = (d * d + s.astype(np.float64)).astype(np.float32)
    return s.argmin(1)


def _train(base, M, iters, train_max, seed):
    n, dim = base.shape
    ns = min(n, train_max)
    xs = base[(np.arange(ns) * n) // ns].astype(np.float32)
    acc = np.zeros(dim)
    for row in xs:
        acc += row
    cent = (acc / ns).astype(np.float32)
    offs = [(i * dim) // M for i in range(M + 1)]
    piv = np.zeros((256, dim), np.float32)
    codes = np.empty((n, M), np.uint8)
    for m in range(M):
        a, b = offs[m], offs[m + 1]
        for c in range(256):
            piv[c, a:b] = xs[_rng(seed, 12 + m, c) % ns, a:b] - cent[a:b]
        x = xs[:, a:b] - cent[a:b]
        for it in range(iters):
            near = _nearest(x, piv[:, a:b])
            for c in range(256):
                rows = np.nonzero(near == c)[0]
                if rows.size == 0:
                    piv[c, a:b] = xs[_rng(seed, 400 + m, it * 256 + c) % ns, a:b] - cent[a:b]
                    continue
                s = np.zeros(b - a)
                for r in rows:
                    s += xs[r, a:b].astype(np.float64) - cent[a:b].astype(np.float64)
                piv[c, a:b] = (s / rows.size).astype(np.float32)
        codes[:, m] = _nearest(base[:, a:b].astype(np.float32) - cent[a:b], piv[:, a:b])
    return cent, piv, codes


# chunk widths 1, 2, 3 and 4 mixed, 8, 16; rows below one wave and one segment (4096), just
# past it, and more rows than the sample; few values, so that pivots repeat and lose their rows
@pytest.mark.parametrize("dtype, n, dim, M, train_max, high", [
    ("uint8", 60, 8, 8, 1 << 18, 256), ("uint8", 4099, 20, 6, 1 << 18, 256), ("int8", 1500, 16, 8, 1000, 256),
    ("float32", 4101, 8, 4, 1 << 18, 256), ("float32", 900, 32, 2, 1 << 18, 256), ("uint8", 1025, 16, 2, 1 << 18, 3),
    ("float32", 2000, 12, 3, 1999, 2),
])
def test_tables_and_codes(lib, dtype, n, dim, M, train_max, high):
    print(f"[gpu] PQ training {dtype} n={n} dim={dim} M={M}", flush=True)
    rng = np.random.default_rng(n)
    base = rng.integers(0, high, (n, dim))
    if dtype == "float32":
        base = base + (rng.standard_normal((n, dim)) if high > 2 else 0)
    base = np.ascontiguousarray(base - (128 if dtype == "int8" else 0)).astype(dtype)
    L = lib.load()
    p = lib.default_build_params()
    p.R, p.L, p.num_chunks, p.kmeans_iters, p.pq_train_max, p.passes, p.seed = 8, 16, M, 3, train_max, 1, 77
    code = {"uint8": lib.QV_UINT8, "int8": lib.QV_INT8, "float32": lib.QV_FLOAT}[dtype]
    db = lib.DeviceBuffer(base.nbytes).upload(base)
    h = C.c_void_p()
    lib.check(L.qv_build_index_gpu(db.ptr, code, n, dim, C.byref(p), 0, C.byref(h)))
    codes, cent, piv = np.empty((n, M), np.uint8), np.empty(dim, np.float32), np.empty((256, dim), np.float32)
    lib.check(L.qv_index_copy_out(h, None, codes.ctypes.data, cent.ctypes.data, piv.ctypes.data, None))
    L.qv_index_close(h)
    want = _train(base, M, 3, train_max, 77)
    np.testing.assert_array_equal(cent, want[0])
    np.testing.assert_array_equal(piv, want[1])
    np.testing.assert_array_equal(codes, want[2])

"""The GPU builder's graph against a Python restatement of batched Vamana
insertion over the oracle's search: candidates sorted by (distance, id) and
deduplicated, RobustPrune, reverse edges with slack, and the final fold of the
slack.  Rows hold small whole numbers (float rows too), so every exact distance
is the same in any order of additions, and graphs are compared edge by edge."""
from __future__ import annotations

import ctypes as C
import math

import numpy as np
import pytest

import qv_oracle as O

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


def _capacity(words, R, lds=160 * 1024):
    """The candidates a prune keeps: four (two) prunes' rows, keys and lists per CU."""
    s4 = (words + 3) // 4
    stride = 4 * (s4 + 1 - s4 % 2)
    size = lambda c: ((12 * c + 15) // 16 * 16 + 4 * stride + max(4 * c * stride, 4096) + 4 * R + 1023) // 1024 * 1024
    c = 256
    while c > 192 and lds // size(c) < 4:
        c -= 8
    if lds // size(c) < 4:
        c = 256
        while c > 64 and lds // size(c) < 2:
            c -= 8
    return c


class Builder:
    def __init__(self, base, R, alpha, capacity):
        self.x, self.R, self.alpha, self.cap = base.astype(np.float64), R, np.float32(alpha), capacity
        self.P = math.ceil(0.3 * R)
        n = base.shape[0]
        self.nbr, self.pend = [[] for _ in range(n)], [[] for _ in range(n)]

    def dist(self, a, b):
        return np.float32(((self.x[a] - self.x[b]) ** 2).sum())

    def prune(self, p, cand):
        keys = sorted({(self.dist(p, c), c) for c in cand[:512] if c != p})[:self.cap]
        self.pend[p] = []
        if len(keys) <= self.R:
            self.nbr[p] = [c for _, c in keys]
            return
        out, alive = [], keys
        while alive and len(out) < self.R:
            _, i = alive[0]
            out.append(i)
            alive = [(d, j) for d, j in alive[1:] if not self.alpha * self.dist(i, j) <= d]
        self.nbr[p] = out

    def insert(self, batch, expanded):
        for p, e in zip(batch, expanded):
            self.prune(p, e[:256] + self.nbr[p] + self.pend[p])
        runs = {}
        for t, s in sorted((t, p) for p in batch for t in self.nbr[p]):
            runs.setdefault(t, []).append(s)
        marked = []
        for t, run in runs.items():
            new = [s for s in run if s not in self.nbr[t] and s not in self.pend[t]]
            room = self.R - len(self.nbr[t])
            if len(new) > room + self.P - len(self.pend[t]):
                marked.append(t)
            else:
                self.nbr[t] += new[:room]
                self.pend[t] += new[room:]
        for t in marked:
            self.prune(t, self.nbr[t] + self.pend[t] + runs[t][:512 - self.R - self.P])

    def fold(self):
        for p, e in enumerate(self.pend):
            if e:
                self.prune(p, self.nbr[p] + e)


# row widths: in registers (8, 24 and 32 pieces of 16 bytes, full and not) and past them, capacities
# below 256; degrees from 1 to the limit; beams whose expansions fill one candidate per thread and more
@pytest.mark.parametrize("dtype, n, dim, M, R, L, passes", [
    ("uint8", 500, 128, 8, 16, 40, 2), ("int8", 300, 20, 4, 3, 12, 1), ("uint8", 400, 4, 2, 1, 8, 1),
    ("uint8", 700, 132, 11, 64, 300, 1), ("float", 400, 96, 12, 12, 30, 2), ("float", 300, 100, 10, 9, 24, 1),
    ("float", 350, 36, 4, 128, 250, 1), ("float", 600, 200, 20, 30, 240, 1),
])
def test_graph(lib, dtype, n, dim, M, R, L, passes):
    print(f"[gpu] graph {dtype} n={n} dim={dim} R={R} L={L}", flush=True)
    rng = np.random.default_rng(n)
    np_type = {"uint8": np.uint8, "int8": np.int8, "float": np.float32}[dtype]
    code = {"uint8": lib.QV_UINT8, "int8": lib.QV_INT8, "float": lib.QV_FLOAT}[dtype]
    base = (rng.integers(0, 12, (8, dim))[rng.integers(0, 8, n)] + rng.integers(0, 6, (n, dim))).astype(np_type)
    Lb = lib.load()
    p = lib.default_build_params()
    p.R, p.L, p.num_chunks, p.kmeans_iters, p.passes, p.seed = R, L, M, 2, passes, 5
    db = lib.DeviceBuffer(base.nbytes).upload(base)
    h = C.c_void_p()
    lib.check(Lb.qv_build_index_gpu(db.ptr, code, n, dim, C.byref(p), 0, C.byref(h)))
    info = lib.IndexInfo()
    lib.check(Lb.qv_index_get_info(h, C.byref(info)))
    pages, codes = np.empty(info.num_pages * 4096, np.uint8), np.empty((n, M), np.uint8)
    cent, piv, offs = np.empty(dim, np.float32), np.empty((256, dim), np.float32), np.empty(M + 1, np.int32)
    lib.check(Lb.qv_index_copy_out(h, pages.ctypes.data, codes.ctypes.data, cent.ctypes.data, piv.ctypes.data,
                                   offs.ctypes.data))
    Lb.qv_index_close(h)
    host = O.HostIndex.from_arrays(code, dim, n, R, int(info.enter_point), pages.copy(), codes, cent, piv, offs)
    got = [host.neighbors(v).tolist() for v in range(n)]

    words = dim * base.itemsize // 4
    b = Builder(base, R, 1.2, _capacity(words, R))
    order = list(range(n))
    for i in range(n - 1, 0, -1):
        j = _rng(5, 21, i) % (i + 1)
        order[i], order[j] = order[j], order[i]

    def write(v):
        rec = host.node_record(v)[dim * base.itemsize:].view(np.uint32)
        rec[0] = len(b.nbr[v])
        rec[1:1 + len(b.nbr[v])] = b.nbr[v]

    for v in range(n):
        write(v)
    for ps in range(passes):
        b.alpha = np.float32(1.0 if passes == 2 and ps == 0 else 1.2)
        done, size = 0, 1 if ps == 0 else 1024
        while done < n:
            batch = order[done:done + min(size, 1024)]
            b.insert(batch, [O.search_trace(host, base[v].astype(np.float32), 1, L)[4] for v in batch])
            for v in range(n):
                write(v)
            done, size = done + len(batch), size * 2
        b.fold()
        for v in range(n):
            write(v)
    assert got == b.nbr

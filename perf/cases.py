"""The calls whose time counts: searches, index construction and exact ground truth.

Sizes, data and options are those of bench.py's workloads, the tests and the
command line's defaults (Vamana R = 64, L = 100, alpha 1.2, PQ 32 x 256 for
8-bit vectors of 128 dimensions and 48 x 256 for float vectors of 96; top-10;
pipe width 2; the seeded Gaussian mixture as data).  Every case is one call
through the C ABI as the Python binding declares it, with device buffers or,
where a case says so, host arrays.
"""
from __future__ import annotations

import ctypes as C
import math
import sys
from pathlib import Path

import numpy as np
import torch

sys.path.insert(0, str(Path.cwd() / "quiver-ae_amd"))

from quiver import _lib  # noqa: E402

_TORCH = {"uint8": torch.uint8, "int8": torch.int8, "float": torch.float32}
_CODE = {"uint8": _lib.QV_UINT8, "int8": _lib.QV_INT8, "float": _lib.QV_FLOAT}
_BYTES = {"uint8": 1, "int8": 1, "float": 4}
_QUERY_ROW = 1 << 40  # queries: rows of the mixture far beyond the base rows


def _search(name, n, nq, ef, *, dim=128, dtype="uint8", R=64, M=32, k=10, pipe=2, policy="none", table=True,
            host=False):
    return dict(name=name, kind="search", n=n, dim=dim, dtype=dtype, R=R, M=M, nq=nq, k=k, ef=ef, pipe=pipe,
                policy=policy, table=table, host=host)


def _build(name, n, *, dim=128, dtype="uint8", R=64, L=100, M=32):
    return dict(name=name, kind="build", n=n, dim=dim, dtype=dtype, R=R, L=L, M=M)


def _truth(name, n, nq, *, dim=128, dtype="uint8", k=10):
    return dict(name=name, kind="truth", n=n, dim=dim, dtype=dtype, nq=nq, k=k)


def listed():
    return [
        # one user's question at a time, at Recall@10 of about 0.90
        _search("one query", 1_000_000, 1, 208),
        # a service's small batch of float vectors, queries and results in host memory
        _search("16 float queries", 300_000, 16, 96, dim=96, dtype="float", M=48, host=True),
        # a larger online batch with the command line's default early exit
        _search("256 queries, gpruning", 500_000, 256, 256, policy="gpruning", table=False),
        # one query file of a benchmark, device-resident, without the neighbour code table
        _search("10k queries", 1_000_000, 10_000, 208, pipe=1, table=False),
        # the same over float vectors at their Recall@10 of 0.90
        _search("10k float queries", 1_000_000, 10_000, 96, dim=96, dtype="float", M=48),
        # graphs of degree 128, as the published billion-point indexes have, a short beam, host arrays
        _search("5k queries, degree 128", 300_000, 5_000, 64, R=128, table=False, host=True),
        # a top-100 over int8 vectors of 100 dimensions: chunks of three and four dimensions
        _search("top-100 int8, ragged", 200_000, 3_000, 256, dim=100, dtype="int8", R=48, k=100, table=False),
        # the throughput benchmark: a long stream of queries in one call over the largest index
        _search("stream of queries", 4_000_000, 100_000, 240),
        # index construction over a shard's worth of 8-bit and of float vectors
        _build("build uint8", 250_000),
        _build("build float", 100_003, dim=96, dtype="float", M=48),
        # exact nearest neighbours, which recall is measured against
        _truth("truth uint8", 1_000_000, 10_000),
        _truth("truth float", 500_001, 2_001, dim=96, dtype="float"),
    ]


def _spread(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    shape = rng.choice([("uint8", 128, 32), ("uint8", 128, 32), ("float", 96, 48), ("int8", 128, 32),
                        ("int8", 100, 32), ("uint8", 100, 25)])
    dtype, dim, M = shape
    kind = rng.choice(["search"] * 7 + ["build", "build", "truth", "truth"])
    if kind == "build":
        R = rng.choice([32, 64, 64, 100])
        c = _build("", _spread(rng, 20_000, 250_000), dim=dim, dtype=dtype, R=R, L=max(R, rng.choice([64, 100])), M=M)
    elif kind == "truth":
        c = _truth("", _spread(rng, 20_000, 1_000_000), _spread(rng, 100, 10_000 if dtype != "float" else 2_500),
                   dim=dim, dtype=dtype, k=rng.choice([1, 10, 10, 16, 50]))
    else:
        R = rng.choice([32, 64, 64, 64, 96, 128])
        big = R > 64
        k = rng.choice([1, 10, 10, 10, 20, 100])
        c = _search("", _spread(rng, 30_000, 200_000 if big else 1_000_000), _spread(rng, 1, 20_000),
                    max(k, _spread(rng, 32, 448)), dim=dim, dtype=dtype, R=R, M=M, k=k, pipe=rng.choice([1, 2, 2, 4]),
                    policy=rng.choice(["none", "none", "gpruning"]),
                    table=not big and M in (32, 48) and rng.random() < 0.5, host=rng.random() < 0.4)
    del c["name"]
    return c


class _Index:
    """A handle, closed with its owner."""

    def __init__(self, handle):
        self.h = handle

    def __del__(self):
        if self.h:
            _lib.load().qv_index_close(self.h)
            self.h = None


def _mixture(case, seed, first, rows):
    """Rows of the seeded mixture as a device tensor (int8: the uint8 mixture shifted by -128)."""
    flt = case["dtype"] == "float"
    mix = _lib.Mixture(seed + 1, max(16, case["n"] // 1024), case["dim"], _lib.QV_FLOAT if flt else _lib.QV_UINT8,
                       32.0, 224.0, 1.0 if flt else 20.0, 1)
    t = torch.empty((rows, case["dim"]), dtype=torch.float32 if flt else torch.uint8, device="cuda")
    torch.cuda.synchronize()
    _lib.check(_lib.load().qv_mixture_fill_device(C.byref(mix), first, rows, t.data_ptr(), 0))
    if case["dtype"] == "int8":
        t = (t.to(torch.int16) - 128).to(torch.int8)
    torch.cuda.synchronize()
    return t


def _params(case, seed):
    p = _lib.default_build_params()
    p.R, p.num_chunks, p.seed = case["R"], case["M"], seed + 7
    p.L = case.get("L", max(100, case["R"]))
    return p


def _built(case, base, params):
    h = C.c_void_p()
    _lib.check(_lib.load().qv_build_index_gpu(base.data_ptr(), _CODE[case["dtype"]], case["n"], case["dim"],
                                              C.byref(params), 0, C.byref(h)))
    return _Index(h)


def prepare(case, seed):
    base = _mixture(case, seed, 0, case["n"])
    s = {"case": case}
    if case["kind"] == "build":
        s["base"], s["params"] = base, _params(case, seed)
        return s
    nq, k = case["nq"], case["k"]
    q = _mixture(case, seed, _QUERY_ROW, nq).float().contiguous()
    host = case.get("host", False)
    where = "cpu" if host else "cuda"
    s["q"] = q.to(where)
    s["ids"] = torch.zeros((nq, k), dtype=torch.int32, device=where)
    s["dists"] = torch.zeros((nq, k), dtype=torch.float32, device=where)
    if case["kind"] == "truth":
        s["base"] = base
    else:
        s["index"] = _built(case, base, _params(case, seed))
        if case["table"]:
            _lib.check(_lib.load().qv_index_neighbour_codes(s["index"].h, 1))
        o = _lib.default_search_opts()
        o.pipe_width = case["pipe"]
        o.early_exit = _lib.QV_EXIT_GPRUNING if case["policy"] == "gpruning" else _lib.QV_EXIT_NONE
        o.device_buffers = 0 if host else 1
        s["opts"] = o
        s["found"] = torch.zeros(nq, dtype=torch.int32, device=where)
    torch.cuda.synchronize()
    return s


def run(s):
    c, L = s["case"], _lib.load()
    if c["kind"] == "search":
        _lib.check(L.qv_search(s["index"].h, s["q"].data_ptr(), c["nq"], c["dim"], c["k"], c["ef"],
                               C.byref(s["opts"]), s["ids"].data_ptr(), s["dists"].data_ptr(), s["found"].data_ptr(),
                               None))
        return {"ids": s["ids"], "dists": s["dists"], "found": s["found"]}
    if c["kind"] == "truth":
        _lib.check(L.qv_ground_truth(s["base"].data_ptr(), _CODE[c["dtype"]], c["n"], c["dim"], s["q"].data_ptr(),
                                     c["nq"], c["k"], s["ids"].data_ptr(), s["dists"].data_ptr(), 0))
        return {"ids": s["ids"], "dists": s["dists"]}
    # build, then the index as a program takes it out of the handle to keep it
    index = _built(c, s["base"], s["params"])
    info = _lib.IndexInfo()
    _lib.check(L.qv_index_get_info(index.h, C.byref(info)))
    pages = np.empty(info.num_pages * 4096, np.uint8)
    codes = np.empty((c["n"], c["M"]), np.uint8)
    centroid = np.empty(c["dim"], np.float32)
    pivots = np.empty((256, c["dim"]), np.float32)
    _lib.check(L.qv_index_copy_out(index.h, pages.ctypes.data, codes.ctypes.data, centroid.ctypes.data,
                                   pivots.ctypes.data, None))
    return {"pages": pages, "codes": codes, "centroid": centroid, "pivots": pivots, "medoid": int(info.enter_point)}


def work(case):
    n, dim, sz = case["n"], case["dim"], _BYTES[case["dtype"]]
    if case["kind"] == "truth":
        nq, k = case["nq"], case["k"]
        return {"bytes": n * dim * sz + nq * dim * 4 + nq * k * 8, "flops": 2 * n * nq * dim}
    R, M = case["R"], case["M"]
    record = dim * sz + 4 + 4 * R
    if case["kind"] == "search":
        # about 1.1 ef expansions a query (a third of them with the early exit, which
        # stops far from convergence); each reads its record and its neighbours' codes
        hops = case["nq"] * (0.35 if case["policy"] == "gpruning" else 1.1) * case["ef"]
        lut = 3 * 256 * dim
        return {"bytes": hops * (record + R * M) + case["nq"] * (4 * dim + 8 * case["k"] + 4),
                "flops": hops * (R * M + 3 * dim) + case["nq"] * lut}
    # Lloyd iterations over the training sample, the codes, and two passes of
    # insertion: a beam search of width L and a prune per point
    train = 15 * min(n, 262144) + n
    hops = 2 * n * 1.1 * case["L"]
    return {"bytes": n * dim * sz + hops * (record + R * M) + n * (record + M),
            "flops": train * 256 * dim * 3 + hops * (R * M + 3 * dim)}


def tolerance(case):
    # Searches and builds are whole numbers (ids, codes, links) and distances
    # whose order of additions is fixed; 8-bit distances are whole numbers.
    # A float ground-truth distance is a 32-bit sum of 96 squares: in another
    # order of additions it is off by about 1e-7, and near ties may swap.
    if case["kind"] == "truth" and case["dtype"] == "float":
        return {"rel": 5e-7, "max": 4e-6, "differ": 1e-4}
    return "exact"


def exact(case, seed):
    """Ground truth by float64 products; a search's or a build's outputs have no
    value of their own in 64 bits."""
    if case["kind"] != "truth":
        return None
    s = prepare(case, seed)
    base, q = s["base"].double(), s["q"].double()
    norms = (base * base).sum(1)
    out = []
    for at in range(0, case["nq"], 500):
        part = q[at:at + 500]
        d = (part * part).sum(1, keepdim=True) + norms[None, :] - 2.0 * (part @ base.T)
        out.append(torch.topk(d, min(case["k"], case["n"]), dim=1, largest=False, sorted=True).values)
    return {"ids": None, "dists": torch.cat(out)}

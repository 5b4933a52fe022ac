"""The per-query-LUT search as a workgroup of three waves (one owns the beam,
two read nodes and sum distances for it) against the oracle, bit for bit:
query copies that share their LDS with the answers (dim <= 128) and that do
not, both code row lengths, chunks of uneven width, every pipe-lane regime
(one lane, two with guesses, more without), fewer queries than lanes and more
than the device holds at once."""
from __future__ import annotations

import ctypes as C

import numpy as np
import pytest

import qv_oracle as O

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def indexes(tmp_path_factory):
    import quiver
    from quiver import _lib

    if _lib.device_count() == 0:
        pytest.skip("no GPU")
    built = {}

    def get(dtype, dim, M, R):
        key = (dtype, dim, M, R)
        if key not in built:
            d = tmp_path_factory.mktemp("team")
            sigma = {} if dtype == "uint8" else {"sigma": 1.0}
            base = quiver.mixture(2500, dim, data_type=dtype, num_centers=20, seed=9, **sigma)
            q = quiver.mixture(1500, dim, data_type=dtype, num_centers=20, seed=9, first_row=1 << 30, **sigma)
            quiver.build_index(base, d / "i", R=R, L=max(40, R), num_chunks=M, threads=0)
            host = O.HostIndex.from_files(d, "uint8" if dtype == "uint8" else "float")
            built[key] = (d, host, q)
        return built[key]

    return get


@pytest.mark.parametrize("dtype, dim, M, R", [("uint8", 128, 32, 64), ("uint8", 132, 32, 24), ("uint8", 100, 48, 33),
                                              ("float", 96, 48, 32), ("float", 160, 48, 16), ("float", 36, 32, 1)])
@pytest.mark.parametrize("pipe, nq, ef, k, policy", [(1, 1, 64, 10, "none"), (2, 3, 65, 1, "none"),
                                                     (2, 1500, 100, 64, "gpruning"), (3, 40, 256, 65, "none"),
                                                     (16, 40, 448, 10, "gpruning"), (1, 300, 257, 100, "gpruning")])
def test_team_kernel(indexes, dtype, dim, M, R, pipe, nq, ef, k, policy):
    import quiver

    print(f"[gpu] team kernel {dtype} d={dim} M={M} R={R} pipe={pipe} nq={nq} ef={ef} k={k} {policy}", flush=True)
    d, host, q = indexes(dtype, dim, M, R)
    q = q[:nq]
    index = quiver.IndexQuiver(d, data_type=dtype, pipe_width=pipe, search_kernel="lut")
    ids, dists = index.search(q, topk=k, ef_search=ef, early_exit_policy=policy)
    index.close()
    assert index.last_report["kernel"] == 1
    want = O.search(host, q.astype(np.float32), k, ef, pipe_width=pipe,
                    early_exit=O.EXIT_GPRUNING if policy == "gpruning" else O.EXIT_NONE)
    np.testing.assert_array_equal(ids, want[0])
    np.testing.assert_array_equal(dists, want[1])


@pytest.mark.parametrize("dtype, dim, M, ef, k, per_cu", [
    ("uint8", 192, 48, 200, 10, 3), ("float", 192, 48, 256, 10, 3), ("uint8", 256, 32, 448, 10, 4),
    ("uint8", 132, 48, 256, 10, 3), ("float", 640, 32, 200, 10, 4), ("float", 144, 48, 65, 1, 3),
    # a large top-k: the team while it holds as many, one wave per query where that holds three for two, and the
    # team again where both hold two (the runtime counts three)
    ("float", 96, 48, 256, 112, 3), ("float", 96, 48, 256, 113, 3), ("uint8", 100, 48, 200, 150, 3),
    ("float", 96, 48, 256, 160, 3), ("float", 96, 48, 256, 161, 3), ("uint8", 132, 48, 256, 113, 3),
])
def test_full_device(indexes, dtype, dim, M, ef, k, per_cu):
    """More queries than the device holds: as many on a CU as with one wave per query, every one right."""
    import quiver
    from quiver import _lib

    print(f"[gpu] full device {dtype} d={dim} M={M} ef={ef} k={k}", flush=True)
    d, host, q = indexes(dtype, dim, M, 16)
    cus = C.c_int32()
    _lib.check(_lib.load().qv_device_info(0, C.create_string_buffer(64), 64, C.byref(cus), C.byref(C.c_int64())))
    index = quiver.IndexQuiver(d, data_type=dtype, pipe_width=1, search_kernel="lut")
    ids, dists = index.search(q, topk=k, ef_search=ef, early_exit_policy="none")
    index.close()
    assert index.last_report["num_blocks"] == min(per_cu * cus.value, len(q))
    want = O.search(host, q.astype(np.float32), k, ef, early_exit=O.EXIT_NONE)
    np.testing.assert_array_equal(ids, want[0])
    np.testing.assert_array_equal(dists, want[1])


@pytest.mark.parametrize("pipe, nq, k, policy", [(1, 1, 10, "none"), (2, 300, 10, "gpruning"), (5, 40, 100, "none")])
def test_launch_without_evaluators(indexes, pipe, nq, k, policy):
    """A workgroup that lacks its evaluators begins no query (nothing would answer for it): the search fails with that
    cause whichever way its queries are admitted, and nothing is left behind."""
    import quiver
    from quiver import _lib

    print(f"[gpu] team kernel launched with one wave, pipe={pipe} nq={nq} k={k}", flush=True)
    d, host, q = indexes("uint8", 128, 32, 64)
    q = np.ascontiguousarray(q[:nq], np.float32)
    index = quiver.IndexQuiver(d, data_type="uint8", pipe_width=pipe, search_kernel="lut")
    L = _lib.load()
    L.qv_index_set_team_waves.argtypes, L.qv_index_set_team_waves.restype = [C.c_void_p, C.c_int32], None
    handle = index._library().handle()
    dq, out = _lib.DeviceBuffer(q.nbytes).upload(q), [_lib.DeviceBuffer(nq * k * 4) for _ in range(2)]
    o = _lib.default_search_opts()
    o.pipe_width, o.kernel, o.device_buffers = pipe, _lib.QV_KERNEL_LUT, 1

    def on_device(entry):
        return entry(handle, dq.ptr, nq, q.shape[1], k, 128, C.byref(o), out[0].ptr, out[1].ptr, None, None)

    L.qv_index_set_team_waves(handle, 1)
    with pytest.raises(_lib.QuiverError, match="without a query's evaluator waves"):
        index.search(q, topk=k, ef_search=128, early_exit_policy=policy)
    for admission in (_lib.QV_ADMIT_STREAMING, _lib.QV_ADMIT_BATCH, _lib.QV_ADMIT_STATIC):
        o.admission = admission
        assert on_device(L.qv_search) == _lib.QV_EHIP
    assert on_device(L.qv_search_noalloc) == _lib.QV_EHIP
    L.qv_index_set_team_waves(handle, 0)
    ids, dists = index.search(q, topk=k, ef_search=128, early_exit_policy=policy)
    index.close()
    want = O.search(host, q, k, 128, pipe_width=pipe,
                    early_exit=O.EXIT_GPRUNING if policy == "gpruning" else O.EXIT_NONE)
    np.testing.assert_array_equal(ids, want[0])
    np.testing.assert_array_equal(dists, want[1])
    for b in (dq, *out):
        b.close()

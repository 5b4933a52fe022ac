"""The per-query-LUT search as a workgroup of three waves (one owns the beam,
two read nodes and sum distances for it) against the oracle, bit for bit:
query copies that share their LDS with the answers (dim <= 128) and that do
not, both code row lengths, chunks of uneven width, every pipe-lane regime
(one lane, two with guesses, more without), fewer queries than lanes and more
than the device holds at once."""
from __future__ import annotations

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

"""Nearest-centroid assignment of the device build against the host build:
exact ties (duplicate centroids), one to many centroid splits, counts around
the 32-centroid tiles and rows of very different magnitudes."""
import numpy as np
import pytest

from chimera_amd import capi

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,k,dim,spread", [(40, 1, 128, 0), (40, 40, 128, 0), (33, 31, 64, 6), (700, 513, 96, 0),
                                            (700, 513, 128, 12), (6000, 4099, 128, 0), (20000, 2048, 128, 4)])
def test_labels_equal_the_host_build(chimera_mod, n, k, dim, spread):
    rng = np.random.default_rng(n + k + dim)
    x = rng.standard_normal((n, dim)).astype(np.float32)
    # every third token repeats another one: duplicate centroids and rows
    x[::3] = x[rng.integers(0, n, size=x[::3].shape[0])]
    # half of the rest lies close to others (inside the filter's margin)
    near = np.arange(1, n, 6)
    x[near] = x[rng.integers(0, n, size=near.size)] + np.float32(2e-3) * rng.standard_normal((near.size, dim)).astype(np.float32)
    if spread:
        x *= np.float32(2.0) ** rng.integers(-spread, spread + 1, size=(n, 1))
    lens = np.full(n // 20 + 1, 20, np.int32)
    lens[-1] = n - 20 * (n // 20)
    lens = lens[lens > 0]
    print(f"{n} rows, {k} centroids, dim {dim}, spread {spread}", flush=True)
    ref = chimera_mod._build_index(x, lens.tolist(), k, 1)
    ctx = capi.Context(None, 1, 4, 2, 1, max_batch=1)
    ctx.build(x, lens, k, 1)
    got = ctx.download(fields=("cluster_pos", "inv_list"))
    ctx.close()
    assert np.array_equal(got["cluster_pos"], ref["cluster_pos"])
    assert np.array_equal(got["inv_list"], ref["inv_list"])


# rows of 258 row blocks take one centroid split, so two lists hold a row's
# candidates: half of the repeats each, on either side of 128 and of the 256
# that a list holds (past it, the rows are recomputed exactly)
@pytest.mark.parametrize("repeats", [250, 262, 506, 520])
def test_many_equal_centroids(chimera_mod, repeats):
    n, k, dim = 132_000, 700, 128
    rng = np.random.default_rng(repeats)
    x = rng.standard_normal((n, dim)).astype(np.float32)
    ids = np.asarray(chimera_mod._sample_centroid_ids(n, k), np.int64)
    near = np.setdiff1d(rng.permutation(n)[: n // 2], ids)
    x[near] = x[0] + np.float32(1e-2) * rng.standard_normal((near.size, dim)).astype(np.float32)
    x[ids[rng.permutation(k)[:repeats]]] = x[0]
    lens = np.full(n // 20, 20, np.int32)
    print(f"{repeats} equal centroids of {k}", flush=True)
    ref = chimera_mod._build_index(x, lens.tolist(), k, 1)
    ctx = capi.Context(None, 1, 4, 2, 1, max_batch=1)
    ctx.build(x, lens, k, 1)
    got = ctx.download(fields=("cluster_pos", "inv_list"))
    ctx.close()
    assert np.array_equal(got["cluster_pos"], ref["cluster_pos"])
    assert np.array_equal(got["inv_list"], ref["inv_list"])

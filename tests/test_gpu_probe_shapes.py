"""Labels of the matrix-core probe equal to the exact fp32 kernel's at the row
counts where its work split changes (waves that share 64 rows, one row block
and more), for one and four sampled tiles per group minimum, many and few
sub-lists, and centroid counts that fill no tile."""
import ctypes as C

import numpy as np
import pytest

from chimera_amd import capi

pytestmark = pytest.mark.gpu


def context(k, nprobe, max_rows, seed):
    rng = np.random.default_rng(seed)
    cent = rng.standard_normal((k, 128)).astype(np.float32)
    cent /= np.linalg.norm(cent, axis=1, keepdims=True)
    cent[k // 3] = cent[k // 7]  # an exact tie
    index = {
        "num_embeddings": k, "dimension": 128, "num_clusters": k, "ex_bits": 1, "flips": np.zeros(64, np.uint8),
        "doc_lens": np.array([k], np.int32), "doc_ptrs": np.array([0, k], np.int32),
        "cluster_pos": np.arange(k + 1, dtype=np.uint64), "clustered_codes": np.zeros(k * 16, np.uint8),
        "clustered_factors": np.ones(k, np.float32), "clustered_doc_ids": np.zeros(k, np.int32),
        "token_to_cluster_pos": np.arange(k, dtype=np.uint32), "full_bit_codes": np.zeros(k * 32, np.uint8),
        "full_bit_factors": np.ones(k, np.float32), "rotated_centroids": cent,
    }
    return capi.Context(index, nprobe, nprobe, 1, 1, max_batch=max_rows // 32), cent, rng


def probe(ctx, d_rows, n, nprobe, mode):
    ctx.set_probe_mode(mode)
    d_lab = ctx.empty((n, nprobe), np.uint32)
    capi.check(capi.lib().chimera_probe_device(ctx.handle, C.c_void_p(d_rows.ptr), n, nprobe, C.c_void_p(d_lab.ptr)))
    ctx.synchronize()
    out = d_lab.numpy()
    d_lab.free()
    return out


@pytest.mark.parametrize("k,nprobe", [(1031, 16), (20011, 100), (70001, 8)])
def test_labels_at_the_row_counts_of_the_plan(k, nprobe):
    ctx, cent, rng = context(k, nprobe, 1056, k)
    rows = cent[rng.integers(0, k, size=1056)] + np.float32(0.05) * rng.standard_normal((1056, 128)).astype(np.float32)
    rows[0] = cent[k // 7]
    d_rows = ctx.to_device(rows)
    for n in (1, 31, 32, 33, 63, 64, 65, 128, 255, 256, 257, 511, 512, 513, 1056):
        print(f"k {k}, nprobe {nprobe}, {n} rows", flush=True)
        assert np.array_equal(probe(ctx, d_rows, n, nprobe, 2), probe(ctx, d_rows, n, nprobe, 1)), n
    d_rows.free()
    ctx.close()

"""One context built, searched and rebuilt over indexes of other sizes and
code widths (its memory is reused where it fits): every index equals the host
build, results equal a fresh context's, and no memory is held past the last
index's."""
import numpy as np
import pytest

from chimera_amd import capi, synthetic

pytestmark = pytest.mark.gpu

KEYS = ("cluster_pos", "inv_list", "token_to_cluster_pos", "one_bit_codes", "full_bit_codes", "full_bit_factors",
        "clustered_codes", "clustered_doc_ids", "rotated_centroids")


def test_rebuilds_of_one_context(chimera_mod):
    ctx = capi.Context(None, 8, 60, 20, 3, max_batch=8)
    sizes = [(3000, 2048, 4, 128), (3100, 2048, 4, 128), (200, 40, 7, 96), (6000, 300, 1, 128), (3000, 2048, 4, 128)]
    held = []
    for i, (docs, clusters, ex_bits, dim) in enumerate(sizes):
        w = synthetic.generate(num_docs=docs, num_centres=64, sigma=0.15, nq=8, seed=i, dim=dim, len_lo=1, len_hi=40)
        print(f"build {i}: {docs} docs, {clusters} clusters, ex_bits {ex_bits}, dim {dim}", flush=True)
        ref = chimera_mod._build_index(w.embeddings, w.doc_lens.tolist(), clusters, ex_bits)
        ctx.build(w.embeddings, w.doc_lens, clusters, ex_bits)
        got = ctx.download()
        for key in KEYS:
            assert np.array_equal(np.asarray(got[key]).ravel(), np.asarray(ref[key]).ravel()), (i, key)
        res = ctx.search(w.queries, 10)
        fresh = capi.Context(ref, 8, 60, 20, 3, max_batch=8)
        for a, b in zip(res, fresh.search(w.queries, 10)):
            assert np.array_equal(a, b), i
        fresh.close()
        held.append(ctx.memory_usage())
    assert held[4] <= 1.3 * held[0]
    with pytest.raises(capi.ChimeraError):
        ctx.build(np.zeros((40, 128), np.float32), np.array([40], np.int32), 8, 4)
    assert ctx.memory_usage() == 0
    ctx.close()

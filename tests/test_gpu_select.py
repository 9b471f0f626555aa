"""The refinement selection spread over the GPU (small sub-batches) against
the query-per-block selection and the oracle: list sizes from all candidates
to a few, ties that overflow the list, scores of other magnitudes (past the
histogram's bins) and bucket sizes."""
import numpy as np
import pytest

from chimera_amd import capi, synthetic
from oracle import oracle as orc

pytestmark = pytest.mark.gpu


def corpus(docs, scale, copies, seed):
    w = synthetic.generate(num_docs=docs, num_centres=64, sigma=0.15, nq=9, seed=seed, len_lo=1, len_hi=6)
    emb = w.embeddings * np.float32(scale)
    lens = w.doc_lens.copy()
    if copies:  # the first document again and again: exact score ties
        first = emb[:lens[0]]
        emb = np.concatenate([emb, np.tile(first, (copies, 1))])
        lens = np.concatenate([lens, np.full(copies, lens[0], np.int32)])
    return np.ascontiguousarray(emb), lens, w.queries


@pytest.mark.parametrize("docs,clusters,nprobe,k_refine,scale,copies", [
    (700, 64, 16, 5000, 1.0, 0),         # every candidate listed
    (9000, 64, 32, 40, 1.0, 0),          # a few of many
    (9000, 64, 32, 2500, 1.0, 0),        # more than the groups could prune
    (9000, 64, 32, 500, 1e-9, 0),        # scores below the lowest bin
    (9000, 64, 32, 500, 3e9, 0),         # and above the highest
    (9000, 64, 48, 300, 1.0, 6000),      # ties past the list
    (30000, 4096, 8, 100, 1.0, 0),       # larger buckets
])
def test_refined_lists(chimera_mod, docs, clusters, nprobe, k_refine, scale, copies):
    emb, lens, queries = corpus(docs, scale, copies, docs + k_refine)
    index = chimera_mod._build_index(emb, lens.tolist(), clusters, 2)
    print(f"{lens.size} docs, nprobe {nprobe}, k_refine {k_refine}, scale {scale}", flush=True)
    ctx = capi.Context(index, nprobe, k_refine, min(20, k_refine), 3, max_batch=16, exact=True)
    t = ctx.search_trace(queries, 10)
    one = ctx.search_trace(queries[:1], 10)
    ctx.close()
    oi = orc.Index(index)
    for q in range(queries.shape[0]):
        ref = orc.search(oi, queries[q], nprobe, k_refine, min(20, k_refine), 3, 10)
        n = int(t["refined_count"][q])
        assert n == len(ref["refined_ids"])
        assert np.array_equal(t["refined_ids"][q, :n], ref["refined_ids"])
        if q == 0:
            assert np.array_equal(one["refined_ids"][0, :n], ref["refined_ids"])


# further shapes that take it: larger buckets whose groups cannot prune, and
# more groups than k_refine with lists of 4,096 and of 8,192 keys
@pytest.mark.parametrize("docs,clusters,nprobe,k_refine", [(30000, 4096, 24, 500), (80000, 64, 24, 1100),
                                                           (150000, 64, 24, 2100)])
def test_refined_lists_of_more_documents(chimera_mod, docs, clusters, nprobe, k_refine):
    test_refined_lists(chimera_mod, docs, clusters, nprobe, k_refine, 1.0, 0)

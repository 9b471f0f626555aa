"""MaxSim rescoring at the sizes where its kernels change (documents shared
by four and two waves, a wave per document) and at the edges of the
16-token tiles, against float64. Split fp16 operands keep a product within
2^-21 of |q||x|, so a 32-token sum stays within 32 * 2^-20 of unit vectors'."""
import numpy as np
import pytest

from chimera_amd import capi

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nq,cap", [(1, 1), (1, 9), (2, 256), (3, 171), (7, 292), (2, 1024), (3, 700)])
def test_scores_against_float64(nq, cap):
    rng = np.random.default_rng(nq * 1000 + cap)
    lens = rng.choice([1, 2, 15, 16, 17, 31, 33, 64, 127, 129, 200], size=60)
    lens[7] = 0
    ptrs = np.concatenate([[0], np.cumsum(lens)]).astype(np.int32)
    emb = rng.standard_normal((int(ptrs[-1]), 128)).astype(np.float32)
    emb /= np.linalg.norm(emb, axis=1, keepdims=True)
    q = rng.standard_normal((nq, 32, 128)).astype(np.float32)
    q /= np.linalg.norm(q, axis=2, keepdims=True)
    ids = rng.integers(-1, 61, size=(nq, cap)).astype(np.int32)  # -1 and 60 are no documents
    counts = np.full(nq, cap, np.int32)
    counts[-1] = max(1, cap - 1)
    print(f"{nq} queries, {cap} candidates", flush=True)
    sims = np.einsum("qid,td->qit", q.astype(np.float64), emb.astype(np.float64))
    doc = np.full((nq, 60), -np.inf)
    for d in range(60):
        if lens[d]:
            doc[:, d] = sims[:, :, ptrs[d]:ptrs[d + 1]].max(2).sum(1)
    ctx = capi.Context(None, 1, 1, 1, 1)
    d_emb, d_ptrs = ctx.to_device(emb), ctx.to_device(ptrs)
    got, top, top_scores, top_counts = ctx.maxsim_rescore(d_emb, d_ptrs, q, ids, counts, 5)
    d_emb.free()
    d_ptrs.free()
    ctx.close()
    for i in range(nq):
        valid = (ids[i] >= 0) & (ids[i] < 60)
        want = np.where(valid, doc[i, np.clip(ids[i], 0, 59)], -np.inf)[:counts[i]]
        have = got[i, :counts[i]].astype(np.float64)
        assert np.array_equal(np.isneginf(want), np.isneginf(have))
        fin = np.isfinite(want)
        assert np.abs(want[fin] - have[fin]).max(initial=0.0) <= 32 * 2.0 ** -20
        best = np.sort(have)[::-1][:5]
        assert np.array_equal(top_scores[i, :top_counts[i]].astype(np.float64)[:best.size], best)

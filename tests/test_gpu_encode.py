"""Token encoding on the device against the host encoder, byte for byte, on
tokens at the edges of the rescale search: events at equal times (grid
values, equal magnitudes), zero components, events past the search range,
one dominant component, components too small for exact sums (the sequential
search), and token counts around the 32 tokens of a step."""
import numpy as np
import pytest

from chimera_amd import capi

pytestmark = pytest.mark.gpu


def edge_tokens(dim, n, seed):
    rng = np.random.default_rng(seed)
    x = rng.standard_normal((n, dim)).astype(np.float32)
    kind = np.arange(n) % 8
    x[kind == 1] = rng.integers(-2, 3, size=(int((kind == 1).sum()), dim))        # ties and zeros
    x[kind == 2] = rng.choice([-1.0, 1.0], size=(int((kind == 2).sum()), dim))    # equal magnitudes
    one = np.flatnonzero(kind == 3)
    x[one] = 0.0
    x[one, rng.integers(0, dim, one.size)] = 3.0                                  # one component
    x[kind == 4] *= np.exp(6.0 * rng.standard_normal((int((kind == 4).sum()), dim))).astype(np.float32)
    x[kind == 5] *= np.float32(1e-18)                                             # tiny tokens
    x[kind == 6] = np.round(x[kind == 6] * 4) * np.float32(0.25)
    x[kind == 7] *= np.float32(2.0) ** rng.integers(-30, 1, size=(int((kind == 7).sum()), dim))
    x[np.abs(x).max(1) == 0, 0] = 1.0
    return x


@pytest.mark.parametrize("ex_bits", [1, 2, 3, 4, 5, 6, 7])
@pytest.mark.parametrize("dim,n,plain", [(128, 1000, False), (96, 1025, False), (64, 257, True), (100, 31, True),
                                         (128, 33, True)])
def test_codes_equal_the_host_encoder(chimera_mod, dim, n, plain, ex_bits):
    """plain: no sign flips, so that grid inputs stay on a grid."""
    x = edge_tokens(dim, n, 7 * dim + n + ex_bits)
    flips = np.zeros(64, np.uint8) if plain else np.random.default_rng(n).integers(0, 256, 64).astype(np.uint8)
    rot = chimera_mod._rotate(x, flips)
    keep = np.isfinite(rot).all(1) & (np.abs(rot).max(1) > 0)
    x, rot = np.ascontiguousarray(x[keep]), np.ascontiguousarray(rot[keep])
    n = x.shape[0]
    print(f"dim {dim}, {n} tokens, plain {plain}, ex_bits {ex_bits}", flush=True)
    ctx = capi.Context(None, 2, 4, 2, 1, max_batch=1)
    ctx.build(x, np.array([n], np.int32), 4, ex_bits, centroid_ids=np.arange(4), flips=flips)
    got = ctx.download(fields=("one_bit_codes", "one_bit_factors", "full_bit_codes", "full_bit_factors"))
    ctx.close()
    codes, f1 = chimera_mod._encode_one_bit(rot)
    full, ff = chimera_mod._encode_full(rot, ex_bits)
    assert np.array_equal(got["one_bit_codes"].reshape(n, 2), codes)
    assert np.array_equal(got["one_bit_factors"].view(np.uint32), f1.view(np.uint32))
    bad = np.flatnonzero((got["full_bit_codes"].reshape(n, -1) != full).any(1))
    assert bad.size == 0, f"{bad.size} tokens differ, first {bad[:5]} (kinds {(np.flatnonzero(keep)[bad] % 8)[:5]})"
    assert np.array_equal(got["full_bit_factors"].view(np.uint32), ff.view(np.uint32))

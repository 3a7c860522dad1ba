"""GPU parity of the fp32 attention kernel, which multiplies split operands on the bf16 matrix cores: accuracy against float64 around the
edges of its 32-key tiles and 128-query workgroups, operands that the split does not survive (infinities, NaN, values that round to
bf16 infinity; the kernel computes those queries again with the fp32 instruction) and scales of either sign."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def exact(q, k, v, scale, causal=False, mask=None):
    q, k, v = (t.astype(np.float64).transpose(0, 2, 1, 3) for t in (q, k, v))
    with np.errstate(invalid="ignore"):
        s = q @ k.transpose(0, 1, 3, 2) * scale
        if mask is not None:
            s = s + (mask[:, None, None, :].astype(np.float64) - 1) * 1e9
        if causal:
            s = np.where(np.triu(np.ones(s.shape[-2:], bool), 1), -np.inf, s)
        w = np.exp(s - s.max(-1, keepdims=True))
        return ((w / w.sum(-1, keepdims=True)) @ v).transpose(0, 2, 1, 3)


def qkv(seed, B, S, H, D):
    rng = np.random.default_rng(seed)
    return [rng.standard_normal((B, S, H, D)).astype(np.float32) for _ in range(3)]


@pytest.mark.parametrize("D", [32, 64, 128])
@pytest.mark.parametrize("S", [1, 31, 32, 33, 64, 65, 127, 129, 300])
@pytest.mark.parametrize("causal", [False, True])
def test_error_against_float64(backend, D, S, causal):
    """A weight is off by the error of its score, 2^-24 times a random walk of sqrt(6 D / 16) roundings at the size of a score (about
    1, at most 6) plus the rounding of the exponent; the sum over keys walks sqrt(6 S / 16) steps."""
    q, k, v = qkv(S + D, 2, S, 3, D)
    mask = (np.arange(S)[None] < np.array([[S], [max(1, S - 5)]])).astype(np.float32)
    bound = 2.0 ** -24 * (6 + np.sqrt(6 * D / 16) + np.sqrt(6 * S / 16))
    for m in (None, mask):
        y = backend.attention.flash_attention2(q, k, v, 3, D, mask=m, causal=causal)
        ref = exact(q, k, v, D ** -0.5, causal, m)
        assert np.linalg.norm(y - ref) < bound * np.linalg.norm(ref)


@pytest.mark.parametrize("D", [32, 64, 128])
def test_weights_keep_the_precision_of_their_exponents(backend, D):
    """100 keys, scores around 1: the exponents of the weights that count are a few units at most, rounded there (about 2^-24), beside the
    scores' walk with steps of half a rounding.  Measured 2.0e-7, 2.5e-7 and 3.1e-7; exponents formed 24 higher give 4.1e-7 to 4.8e-7."""
    q, k, v = qkv(D + 100, 2, 100, 4, D)
    for mask in (None, np.ones((2, 100), np.float32)):
        y, ref = backend.attention.flash_attention2(q, k, v, 4, D, mask=mask), exact(q, k, v, D ** -0.5)
        assert np.linalg.norm(y - ref) < 2.0 ** -24 * (2.2 + 0.5 * np.sqrt(6 * D / 16)) * np.linalg.norm(ref)


@pytest.mark.parametrize("D", [32, 64, 128])
@pytest.mark.parametrize("causal", [False, True])
def test_operands_that_do_not_split(backend, D, causal):
    S, H = 150, 2
    q, k, v = qkv(D, 1, S, H, D)
    q[..., 0] = np.abs(q[..., 0]) + 0.1
    k[0, 3, 0, 0] = -np.inf                       # a score of -infinity: no weight
    v[0, 40, 1, 5] = np.inf                       # an infinite value: that dimension of every query that sees it
    v[0, 41, 1, 6] = np.finfo(np.float32).max     # rounds to bf16 infinity
    q[0, 9, 0, 2] = np.nan                        # one query
    y = backend.attention.flash_attention2(q, k, v, H, D, causal=causal)
    ref = exact(q, k, v, D ** -0.5, causal)
    if causal:                                    # queries in front of the infinite value: 0 times infinity in the oracle's product
        y[0, :40, 1, 5] = ref[0, :40, 1, 5] = 0.0
    np.testing.assert_array_equal(np.isnan(y), np.isnan(ref))
    np.testing.assert_array_equal(np.isinf(y), np.isinf(ref))
    ok = np.isfinite(ref)
    small = ok & (np.abs(ref) < 1e3)
    assert np.linalg.norm(y[small] - ref[small]) < 1e-6 * np.linalg.norm(ref[small])
    assert np.allclose(y[ok & ~small], ref[ok & ~small], rtol=1e-5, atol=0)


@pytest.mark.parametrize("scale", [-0.2, 0.0, 0.5])
def test_scales(backend, scale):
    q, k, v = qkv(7, 2, 70, 2, 64)
    for causal in (False, True):
        y = backend.attention.flash_attention2(q, k, v, 2, 64, scale=scale, causal=causal)
        ref = exact(q, k, v, scale, causal)
        assert np.linalg.norm(y - ref) < 1e-6 * np.linalg.norm(ref)


def clear_rows(q, k, scale, gap):
    """Queries whose best key is ahead of the second by more than `gap`: the output is that key's value."""
    s = np.einsum("bqhd,bkhd->bqhk", q.astype(np.float64), k.astype(np.float64)) * scale
    top = np.sort(s, -1)
    return top[..., -1] - top[..., -2] > gap


@pytest.mark.parametrize("D", [32, 64, 128])
@pytest.mark.parametrize("mag", [900.0, 2e4, 5e4])
def test_large_scores(backend, D, mag):
    """Scores of 2^20 and far beyond, where a unit in the last place is many powers of two of a weight: the largest weight is 1 all the
    same, with and without a mask that excludes nothing.  (Products round to 2^-24 of about mag^2 each: the best key is told from
    the second where 1e-4 of that lies between them.)"""
    S, H = 70, 3
    q, k, v = qkv(D, 2, S, H, D)
    q, k = q * np.float32(mag), k * np.float32(mag)
    clear = clear_rows(q, k, D ** -0.5, 1e-4 * mag * mag)
    assert clear.mean() > 0.9
    ref = exact(q, k, v, D ** -0.5)
    for mask in (None, np.ones((2, S), np.float32)):
        y = backend.attention.flash_attention2(q, k, v, H, D, mask=mask)
        np.testing.assert_allclose(y[clear], ref[clear], rtol=1e-6, atol=1e-7)
    k[0, 3, 0, 0] = np.inf                        # head 0 of batch entry 0 once more with the fp32 instruction
    q[0, :, 0, 0] = -np.abs(q[0, :, 0, 0])        # a score of -infinity: no weight
    y, kk = backend.attention.flash_attention2(q, k, v, H, D), k.copy()
    kk[0, 3, 0, 0] = 1e30
    clear = clear_rows(q, kk, D ** -0.5, 1e-4 * mag * mag)
    ref = exact(q, kk, v, D ** -0.5)
    np.testing.assert_allclose(y[clear], ref[clear], rtol=1e-6, atol=1e-7)


@pytest.mark.parametrize("scale", [0.0, 1e-38, -3e-39])
def test_scales_next_to_zero_with_large_products(backend, scale):
    q, k, v = qkv(7, 1, 70, 2, 64)
    q, k = q * np.float32(2.0 ** 62), k * np.float32(2.0 ** 60)      # products around 1e38
    for causal in (False, True):
        y = backend.attention.flash_attention2(q, k, v, 2, 64, scale=scale, causal=causal)
        ref = exact(q, k, v, np.float64(np.float32(scale)), causal)
        assert np.linalg.norm(y - ref) < 1e-5 * np.linalg.norm(ref)      # (a scale below the normal numbers has few bits)


@pytest.mark.parametrize("D", [32, 64, 128])
@pytest.mark.parametrize("eq,ek,ev", [(-118, 116, 0), (116, -118, 0), (-125, 124, 0), (0, 0, -112), (0, 0, -120), (-60, 60, -118), (0, 0, 100)])
def test_operands_far_below_one(backend, D, eq, ek, ev):
    """Operands near the smallest normal number, with partners that bring the products back to ordinary size: the bound of
    test_error_against_float64."""
    S, H = 129, 2
    q, k, v = qkv(D - ev - 2 * eq, 2, S, H, D) if ev + 2 * eq < D else qkv(D + 400, 2, S, H, D)
    sq, sk, sv = (np.float32(2.0 ** e) for e in (eq, ek, ev))
    q, k, v = q * sq, k * sk, v * sv
    bound = 2.0 ** -24 * (6 + np.sqrt(6 * D / 16) + np.sqrt(6 * S / 16))
    for causal in (False, True):
        y = backend.attention.flash_attention2(q, k, v, H, D, causal=causal).astype(np.float64) / np.float64(sv)
        ref = exact(q, k, v, D ** -0.5, causal) / np.float64(sv)
        assert np.linalg.norm(y - ref) < bound * np.linalg.norm(ref)


@pytest.mark.parametrize("D", [32, 64, 128])
def test_tiny_weight_of_a_large_value(backend, D):
    """A weight of 2^-122 on a value of 2^110, beside one of 1 on a value of 2^-20.  The products are exact, the score is -85: its weight
    is off by 85 * 2^-24 and the exponent's rounding."""
    S, H = 40, 2
    rng = np.random.default_rng(D)
    q, k, v = np.zeros((1, S, H, D), np.float32), np.zeros((1, S, H, D), np.float32), rng.standard_normal((1, S, H, D)).astype(np.float32)
    q[..., 0], k[..., 0] = 1.0, -2000.0
    k[0, 0, :, 0] = 0.0
    k[0, 33, :, 0] = -85.0
    v[0, 0] *= np.float32(2.0 ** -20)
    v[0, 33] *= np.float32(2.0 ** 110)
    y, ref = backend.attention.flash_attention2(q, k, v, H, D, scale=1.0), exact(q, k, v, 1.0)
    assert np.linalg.norm(y - ref) < 4 * 85 * 2.0 ** -24 * np.linalg.norm(ref)

"""f32 prefill attention on the matrix instructions: query groups of 16 (up to 80 features) or 32, key tiles of 32; by the size of the call (small ones
stay with the kernel that takes a row to a block), and every head size with one, two and four waves to a group forced."""
import numpy as np
import pytest

from rai_amd._lib import RaiHipError
from tests.util import down, rand, up

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def R(hip):
    from rai_amd import ops

    return ops


def reference(q, k, v, scale, causal):
    q, k, v = (t.astype(np.float64) for t in (q, k, v))
    n = q.shape[1] // k.shape[1]
    k, v = np.repeat(k, n, 1), np.repeat(v, n, 1)
    s, size = np.matmul(q, np.swapaxes(k, 2, 3)) * scale, np.matmul(np.abs(q), np.swapaxes(np.abs(k), 2, 3)) * scale
    S, T = s.shape[2:]
    if causal:
        s = np.where(np.arange(T)[None] <= np.arange(T - S, T)[:, None], s, -np.inf)
    p = np.exp(s - s.max(-1, keepdims=True))
    p /= p.sum(-1, keepdims=True)
    # A score's sum is within D + 2 roundings of its absolute sum; twice that error of the largest score (numerator and
    # denominator), and T + 8 roundings of the weighted sum, reach the output relative to sum p |v|.
    rel = 2 * (q.shape[-1] + 2) * 2.0 ** -24 * size.max() + (T + 8) * 2.0 ** -23
    flat = lambda t: np.swapaxes(t, 1, 2).reshape(t.shape[0], S, -1)  # noqa: E731
    with np.errstate(invalid="ignore"):
        return flat(p @ v), rel * flat(p @ np.abs(v))


@pytest.mark.parametrize("causal", [1, 0])
@pytest.mark.parametrize("b,hq,hkv,s,t,d", [(1, 2, 2, 16, 32, 64), (2, 3, 1, 33, 65, 80), (1, 4, 2, 128, 128, 128), (1, 2, 1, 31, 300, 32), (1, 1, 1, 97, 129, 192),
                                            (1, 2, 1, 64, 200, 256), (3, 24, 24, 40, 160, 64), (16, 36, 6, 64, 64, 128), (1, 64, 64, 33, 129, 80),
                                            (1, 64, 16, 32, 65, 64), (16, 36, 6, 64, 64, 64), (2, 64, 64, 31, 80, 32), (1, 64, 8, 33, 300, 128),
                                            (1, 64, 8, 32, 256, 128), (16, 36, 6, 33, 257, 128), (1, 32, 4, 260, 515, 192), (1, 16, 16, 520, 520, 256), (1, 64, 64, 33, 65, 80), (16, 36, 6, 64, 64, 80),
                                            (8, 36, 6, 33, 257, 128), (2, 32, 4, 260, 515, 192)])
def test_against_64_bits(R, b, hq, hkv, s, t, d, causal):
    g = np.random.Generator(np.random.PCG64(b + s))
    q, k, v = rand(g, (b, hq, s, d), "f32"), rand(g, (b, hkv, t, d), "f32"), rand(g, (b, hkv, t, d), "f32")
    want, tol = reference(q, k, v, d ** -0.5, causal)
    got = down(R.attention(up(q, "f32"), up(k, "f32"), up(v, "f32"), d ** -0.5, causal, 1)).astype(np.float64)
    assert np.all(np.abs(got - want) <= tol)


# Head sizes with the waves to a group they come with.
FORMS = [(d, waves) for d in (32, 64, 80, 128, 192, 256) for waves in (1, 2, 4) if waves < 4 or d <= 128]


@pytest.mark.parametrize("causal", [1, 0])
@pytest.mark.parametrize("b,hq,hkv,s,t", [(1, 2, 1, 16, 32), (2, 3, 3, 33, 65), (1, 4, 2, 130, 161), (1, 2, 2, 200, 200)])
@pytest.mark.parametrize("d,waves", FORMS)
def test_every_form_against_64_bits(R, monkeypatch, d, waves, b, hq, hkv, s, t, causal):
    monkeypatch.setenv("RAI_HIP_ATTN_F32", str(waves))   # read per call; refused where it does not apply
    test_against_64_bits(R, b, hq, hkv, s, t, d, causal)


def test_a_form_that_does_not_apply_is_refused(R, monkeypatch):
    g = np.random.Generator(np.random.PCG64(3))
    for waves, s, d in [(4, 64, 256), (3, 64, 64), (1, 15, 64), (1, 64, 48)]:
        q = up(rand(g, (1, 2, s, d), "f32"), "f32")
        monkeypatch.setenv("RAI_HIP_ATTN_F32", str(waves))
        with pytest.raises(RaiHipError):
            R.attention(q, q, q, 0.1, 1, 1)
        monkeypatch.delenv("RAI_HIP_ATTN_F32")
        R.attention(q, q, q, 0.1, 1, 1)


@pytest.mark.parametrize("s,t", [(40, 70), (200, 200)])
@pytest.mark.parametrize("d,waves", FORMS)
def test_infinite_values_with_every_form(R, monkeypatch, d, waves, s, t):
    monkeypatch.setenv("RAI_HIP_ATTN_F32", str(waves))
    test_infinite_values_reach_only_queries_that_see_them(R, s, t, 2, d)


@pytest.mark.parametrize("s,t,n", [(40, 70, 2), (200, 200, 2), (40, 70, 64), (200, 200, 16)])
def test_infinite_values_reach_only_queries_that_see_them(R, s, t, n, d=64):
    g = np.random.Generator(np.random.PCG64(9))
    q, k, v = rand(g, (1, n, s, d), "f32"), rand(g, (1, n, t, d), "f32"), rand(g, (1, n, t, d), "f32")
    clean, tol = reference(q, k, v, d ** -0.5, 1)
    at = t - s // 2
    v[0, 0, at, 5], v[0, 0, t - 1, 7], v[0, 1, at, d - 1] = np.inf, np.nan, -np.inf   # d - 1: the last feature
    got = down(R.attention(up(q, "f32"), up(k, "f32"), up(v, "f32"), d ** -0.5, 1, 1)).astype(np.float64)
    want = clean.copy()
    first = at - (t - s)   # the query at the key's own position
    want[0, first:, 5], want[0, s - 1, 7], want[0, first:, 2 * d - 1] = np.inf, np.nan, -np.inf
    same = np.isfinite(want)
    assert np.array_equal(np.isnan(got), np.isnan(want)) and np.array_equal(got[~same & ~np.isnan(want)], want[~same & ~np.isnan(want)])
    assert np.all(np.abs(got - clean)[same] <= tol[same])


@pytest.mark.parametrize("causal", [1, 0])
@pytest.mark.parametrize("b,hq,hkv,s,t,d", [(1, 64, 8, 16, 63, 80), (1, 65, 13, 16, 63, 80), (1, 1, 1, 16, 64, 64), (2, 3, 1, 17, 95, 32), (1, 4, 2, 16, 1000, 80), (1, 32, 8, 33, 40, 64),
                                            (1, 48, 6, 256, 256, 64), (1, 49, 7, 256, 256, 32), (8, 32, 8, 64, 64, 80), (7, 32, 8, 64, 65, 80), (16, 16, 4, 63, 160, 32)])
def test_around_the_lines_of_the_dispatch(R, b, hq, hkv, s, t, d, causal):
    """A block to a row or tiles; four, two or one wave to a group of 16 rows."""
    test_against_64_bits(R, b, hq, hkv, s, t, d, causal)


def test_few_rows_of_more_keys_than_a_block_holds_are_refused(R):
    q, k = up(np.zeros((1, 1, 16, 32), np.float32), "f32"), up(np.zeros((1, 1, 40000, 32), np.float32), "f32")
    with pytest.raises(RaiHipError):
        R.attention(q, k, k, 0.1, 1, 1)

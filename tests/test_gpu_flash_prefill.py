"""bf16 prefill attention on the matrix instructions: every head size with every number of waves to a query group and both tile
lengths, which the number of groups picks; key counts at and around the ends of tiles, strided operands, scales of any sign."""
import numpy as np
import pytest

from oracle.dtypes import rnd
from tests.util import down, rand, up

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def R(hip):
    from rai_amd import ops

    return ops


def whole(g, shape, step=1.0):
    """Whole multiples of a power of two: sums of their products are exact in f32, in any order."""
    return (g.integers(-4, 5, shape) * step).astype(np.float32)


def reference(q, k, v, scale, causal, f32_scores, rounded=True):
    """The result in 64 bits (scores rounded as the model rounds them) and how far a correct bf16 form may be off.  Scores that are
    rounded are those of whole(): either rounding could turn on the last bit of a sum, and a turned score is far more than the
    arithmetic's own error."""
    q, k, v = (t.astype(np.float64) for t in (q, k, v))
    n = q.shape[1] // k.shape[1]
    k, v = np.repeat(k, n, 1), np.repeat(v, n, 1)
    s, size = np.matmul(q, np.swapaxes(k, 2, 3)), np.matmul(np.abs(q), np.swapaxes(np.abs(k), 2, 3)).max()
    S, T = s.shape[2:]
    if f32_scores:   # a score's f32 sum is within D + 2 roundings of its absolute sum
        off = (q.shape[-1] + 2) * 2.0 ** -24 * size * abs(scale)
        s = s * scale
    else:
        assert size < 2 ** 20 and np.array_equal(s * 4, np.rint(s * 4))
        if rounded:
            s = rnd(rnd(s.astype(np.float32), "bf16") * rnd(np.float32(scale), "bf16"), "bf16").astype(np.float64)
        else:
            s = s * scale
        off = (2 * np.abs(s).max() + 8) * 2.0 ** -24   # the exponent's product with log2(e) and the exponential
    if causal:
        s = np.where(np.arange(T)[None] <= np.arange(T - S, T)[:, None], s, -np.inf)
    p = np.exp(s - s.max(-1, keepdims=True))
    p /= p.sum(-1, keepdims=True)
    flat = lambda t: np.swapaxes(t, 1, 2).reshape(t.shape[0], S, -1)  # noqa: E731
    want = flat(p @ v)
    # scores (numerator and denominator), weights rounded to bf16 (2^-8 at most), f32 sums over the keys; the result's own rounding
    rel = 2 * np.expm1(off) + 2.0 ** -8 + (T + 8) * 2.0 ** -23
    return want, rel * flat(p @ np.abs(v)) * (1 + 2.0 ** -8) + 2.0 ** -8 * np.abs(want) + 1e-30


def operands(g, b, hq, hkv, s, t, d, f32_scores):
    if f32_scores:
        return rand(g, (b, hq, s, d), "bf16"), rand(g, (b, hkv, t, d), "bf16"), rand(g, (b, hkv, t, d), "bf16")
    return whole(g, (b, hq, s, d)), whole(g, (b, hkv, t, d), 0.25), rand(g, (b, hkv, t, d), "bf16")


def check(R, b, hq, hkv, s, t, d, causal, f32_scores, scale=None, transposed=False):
    g = np.random.Generator(np.random.PCG64(b + s + d))
    plain, scale = scale is None, (1 if f32_scores else 3) * d ** -0.5 if scale is None else scale
    q, k, v = operands(g, b, hq, hkv, s, t, d, f32_scores)
    lay = (lambda x: up(np.ascontiguousarray(np.swapaxes(x, 1, 2)), "bf16").transpose(1, 2)) if transposed else (lambda x: up(x, "bf16"))
    want, tol = reference(q, k, v, scale, causal, f32_scores)
    got = down(R.attention(lay(q), lay(k), lay(v), scale, causal, f32_scores)).astype(np.float64)
    assert np.all(np.abs(got - want) <= tol), f"worst {np.max(np.abs(got - want) / tol):.2f} of the bound"
    if plain and t > 16:   # the bound tells scores that are a fiftieth off, and ones that are not rounded, from these
        others = [reference(q, k, v, 1.02 * scale, causal, f32_scores)] + ([] if f32_scores else [reference(q, k, v, scale, causal, 0, False)])
        for other, _ in others:
            assert np.any(np.abs(other - want) > 2 * tol)


# (sequences, query heads, key heads, rows, keys): up to 256 groups of 32 rows, up to 512, 1024, 1536 and beyond 1792; one tile, a last tile
# of one key, of all but one; rows that end inside a group.
SIZES = [(1, 2, 1, 16, 16), (1, 3, 3, 33, 65), (2, 4, 2, 64, 64), (1, 2, 2, 160, 191), (1, 8, 2, 257, 257), (2, 20, 4, 270, 285),
         (3, 40, 40, 140, 150), (2, 64, 8, 300, 300), (7, 64, 64, 97, 129)]


@pytest.mark.parametrize("f32_scores", [0, 1])
@pytest.mark.parametrize("b,hq,hkv,s,t", SIZES)
@pytest.mark.parametrize("d", [32, 64, 80, 128, 192, 256])
def test_forms(R, d, b, hq, hkv, s, t, f32_scores):
    check(R, b, hq, hkv, s, t, d, 1, f32_scores)


@pytest.mark.parametrize("f32_scores", [0, 1])
@pytest.mark.parametrize("b,hq,hkv,s,t", [(1, 3, 3, 33, 95), (3, 40, 40, 140, 150)])
@pytest.mark.parametrize("d", [64, 80, 128, 256])
def test_all_keys_and_strides(R, d, b, hq, hkv, s, t, f32_scores):
    check(R, b, hq, hkv, s, t, d, 0, f32_scores, transposed=True)


@pytest.mark.parametrize("f32_scores", [0, 1])
@pytest.mark.parametrize("scale", [-0.125, 0.0, 0.3])
def test_scales(R, scale, f32_scores):
    check(R, 1, 4, 2, 70, 130, 64, 1, f32_scores, scale=scale)


@pytest.mark.parametrize("f32_scores", [0, 1])
@pytest.mark.parametrize("scale", [0.0, -0.125, 0.25])
def test_scales_keep_what_is_not_a_number(R, scale, f32_scores):
    """Queries and keys with an infinity or a NaN in them: the rows that see one, and no others, are not numbers, at a scale of zero too."""
    g = np.random.Generator(np.random.PCG64(4))
    q, k, v = rand(g, (1, 2, 96, 64), "bf16"), rand(g, (1, 2, 96, 64), "bf16"), rand(g, (1, 2, 96, 64), "bf16")
    q[0, 0, 7, 3], q[0, 0, 40, 63] = np.inf, np.nan
    k[0, 1, 70, 5] = np.nan
    k[0, 1, 80, 6] = np.inf
    got = down(R.attention(up(q, "bf16"), up(k, "bf16"), up(v, "bf16"), scale, 1, f32_scores)).reshape(96, 2, 64)
    lost = np.zeros((96, 2), bool)
    lost[[7, 40], 0] = True
    lost[70:, 1] = True
    if scale:   # a row's infinite scores are of either sign: above all others its weights are not numbers, below them they are zero
        lost[7, 0] = bool((np.sign(k[0, 0, :8, 3]) * np.sign(scale) > 0).any())
    np.testing.assert_array_equal(np.isnan(got).any(-1), lost)
    if scale == 0:
        mean = np.cumsum(v[0].astype(np.float64), 1) / np.arange(1, 97)[:, None]
        keep = ~lost
        want = np.swapaxes(mean, 0, 1)[keep]
        bound = np.swapaxes(np.cumsum(np.abs(v[0].astype(np.float64)), 1) / np.arange(1, 97)[:, None], 0, 1)[keep]
        assert np.all(np.abs(got[keep] - want) <= 2.0 ** -8 * np.abs(want) + 2.0 ** -15 * bound)   # weights of 1: f32 sums, one rounding


def test_more_blocks_than_one_grid_dimension_holds(R):
    """257 x 65528 heads of one block of 256 threads: more than 2^32 threads (the output is 17 GB; whole sequences of it are looked at,
    among them those on both sides of block 2^23 and of block 2^24)."""
    from rai_amd._lib import call

    b, hq, s, d = 257, 65528, 16, 32
    g = np.random.Generator(np.random.PCG64(2))
    q, k, v = rand(g, (1, hq, s, d), "bf16"), rand(g, (b, 1, s, d), "bf16"), rand(g, (b, 1, s, d), "bf16")
    got = R.attention(up(q, "bf16").broadcast_to((b, hq, s, d)), up(k, "bf16"), up(v, "bf16"), d ** -0.5, 1, 1)
    for i in (0, 127, 128, 129, 255, 256):
        want, tol = reference(q, k[i:i + 1], v[i:i + 1], d ** -0.5, 1, 1)
        assert np.all(np.abs(down(got.narrow(0, i, 1)).astype(np.float64) - want) <= tol), i
    del got
    call("rai_hip_trim", 0)

"""Batched products of several steps of K: one to six of them, whole and not, with tiles that end inside a 16-byte piece, a row shorter than one, and
operands that lie among NaNs, of which none may come in."""
import numpy as np
import pytest

from tests.util import down, rand, up

pytestmark = pytest.mark.gpu
U = {"f32": 2.0 ** -24, "bf16": 2.0 ** -8, "f16": 2.0 ** -11}


def among_nans(x, dt, turned):
    """x as a view of a larger tensor of NaNs, its last two axes the other way round in memory if `turned`."""
    x = x.swapaxes(1, 2) if turned else x
    b, r, c = x.shape
    wide = np.full((b, r + 2, c + 12), np.nan, np.float32)
    wide[:, 1:r + 1, 5:c + 5] = x
    t = up(wide, dt).narrow(1, 1, r).narrow(2, 5, c)
    return t.transpose(1, 2) if turned else t


@pytest.mark.parametrize("m,k,n", [(65, 260, 7), (3, 256, 8), (64, 257, 9), (70, 320, 63), (1, 383, 65), (130, 384, 71), (9, 129, 72), (64, 192, 135),
                                   (2, 161, 5), (67, 64, 67), (66, 96, 130), (7, 100, 300)])
@pytest.mark.parametrize("a_t", [False, True])
@pytest.mark.parametrize("b_t", [False, True])
@pytest.mark.parametrize("dt", ["f32", "bf16", "f16"])
def test_steps(hip, dt, a_t, b_t, m, k, n):
    from rai_amd import ops as R

    g = np.random.Generator(np.random.PCG64(m * k + n))
    a, b = rand(g, (3, m, k), dt), rand(g, (3, k, n), dt)
    got = down(R.matmul(among_nans(a, dt, a_t), among_nans(b, dt, b_t))).astype(np.float64)
    a, b = a.astype(np.float64), b.astype(np.float64)
    want = a @ b
    # k products (rounded in f32) and additions of f32 below the sum of magnitudes, one rounding of the result
    assert np.all(np.abs(got - want) <= 2 * (k + 8) * 2.0 ** -24 * (np.abs(a) @ np.abs(b)) + U[dt] * np.abs(want))


@pytest.mark.parametrize("dt", ["bf16", "f16"])
@pytest.mark.parametrize("b_t", [False, True])
def test_large_tiles(hip, dt, b_t):
    """128 x 128 tiles, which 512 of them and a K of 256 take."""
    from rai_amd import ops as R

    g = np.random.Generator(np.random.PCG64(7))
    a, b = rand(g, (60, 257, 325), dt), rand(g, (60, 325, 261), dt)
    got = down(R.matmul(up(a, dt), up(np.ascontiguousarray(b.swapaxes(1, 2)), dt).transpose(1, 2) if b_t else up(b, dt))).astype(np.float64)
    a, b = a.astype(np.float64), b.astype(np.float64)
    want = a @ b
    assert np.all(np.abs(got - want) <= 2 * (325 + 8) * 2.0 ** -24 * (np.abs(a) @ np.abs(b)) + U[dt] * np.abs(want))


@pytest.mark.parametrize("dt", ["bf16", "f16"])
@pytest.mark.parametrize("k,lie", [(257, 257), (264, 267), (129, 129), (104, 107)])
def test_contiguous_along_k_off_boundaries(hip, dt, k, lie):
    """Both operands contiguous along K in rows off 16-byte boundaries: 128 x 128 tiles from K = 256 on, 64 x 64 below; every call the same bits."""
    from rai_amd import ops as R

    g = np.random.Generator(np.random.PCG64(k))
    some = np.arange(130) % 3
    a, b = rand(g, (3, 255, lie), dt), rand(g, (3, 241, lie), dt)
    a[..., k:], b[..., k:] = np.nan, np.nan
    ad, bd = up(a[some], dt).narrow(2, 0, k), up(b[some], dt).narrow(2, 0, k).transpose(1, 2)
    first = down(R.matmul(ad, bd))
    a, b = a[..., :k].astype(np.float64), b[..., :k].astype(np.float64).swapaxes(1, 2)
    want = a @ b
    assert np.all(np.abs(first[:3] - want) <= 2 * (k + 8) * 2.0 ** -24 * (np.abs(a) @ np.abs(b)) + U[dt] * np.abs(want))
    assert np.array_equal(first, first[:3][some])
    for _ in range(4):
        assert np.array_equal(down(R.matmul(ad, bd)), first)

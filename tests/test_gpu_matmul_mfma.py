"""Batched products on the matrix instructions: every layout they take (each operand along K or across it, broadcast and
strided batches, odd sizes, rows that start anywhere), at the edges of tiles and of K tiles."""
import numpy as np
import pytest

from tests.util import down, rand, up

pytestmark = pytest.mark.gpu

# unit roundoff of the result, smallest positive value
ROUND = {"f32": (2.0 ** -24, 2.0 ** -149), "bf16": (2.0 ** -8, 2.0 ** -133), "f16": (2.0 ** -11, 2.0 ** -24)}


@pytest.fixture(scope="module")
def R(hip):
    from rai_amd import ops

    return ops


def check(got, a, b, dt):
    """One rounding to the dtype, and K + 1 roundings of the absolute sum in f32 for the sum in whatever order."""
    a, b = a.astype(np.float64), b.astype(np.float64)
    want, (eps, tiny) = a @ b, ROUND[dt]
    tol = eps * np.abs(want) + tiny + (a.shape[-1] + 1) * 2.0 ** -23 * (np.abs(a) @ np.abs(b))
    assert np.all(np.abs(got.astype(np.float64) - want) <= tol)


@pytest.mark.parametrize("dt", ["f32", "bf16", "f16"])
@pytest.mark.parametrize("a_t,b_t", [(0, 0), (0, 1), (1, 0), (1, 1)])
@pytest.mark.parametrize("batch,m,k,n", [(2, 1, 1, 1), (3, 1, 70, 65), (2, 5, 7, 3), (2, 64, 64, 64), (3, 65, 33, 63), (2, 33, 97, 130),
                                         (2, 31, 129, 8), (5, 70, 200, 66)])
def test_layouts_and_tile_edges(R, dt, a_t, b_t, batch, m, k, n):
    g = np.random.Generator(np.random.PCG64(5))
    a, b = rand(g, (batch, m, k), dt), rand(g, (batch, k, n), dt)
    ad = up(np.swapaxes(a, 1, 2), dt).transpose(1, 2) if a_t else up(a, dt)
    bd = up(np.swapaxes(b, 1, 2), dt).transpose(1, 2) if b_t else up(b, dt)
    check(down(R.matmul(ad, bd)), a, b, dt)


@pytest.mark.parametrize("dt", ["f32", "bf16", "f16"])
@pytest.mark.parametrize("k", [*range(1, 18), 31, 63, 65, 71, 97, 131])
def test_rows_that_end_inside_a_piece(R, dt, k):
    """K along both operands, what lies next to the rows' ends is NaN: none of it is used."""
    g = np.random.Generator(np.random.PCG64(k))
    for m, n, pad in [(3, 2, 1), (70, 5, 9), (33, 65, 16)]:
        a, b = rand(g, (2, m, k + pad), dt), rand(g, (2, n, k + pad), dt)
        a[..., k:], b[..., k:] = np.nan, np.nan
        got = down(R.matmul(up(a, dt).narrow(2, 0, k), up(b, dt).narrow(2, 0, k).transpose(1, 2)))
        check(got, a[..., :k], np.swapaxes(b[..., :k], 1, 2), dt)


@pytest.mark.parametrize("dt", ["bf16", "f16"])
@pytest.mark.parametrize("b_t", [0, 1])
def test_large_tiles(R, dt, b_t):
    """Enough 128 x 128 tiles for that form, ragged in every direction."""
    g = np.random.Generator(np.random.PCG64(6))
    a, b = rand(g, (40, 400, 263), dt), rand(g, (40, 263, 500), dt)
    bd = up(np.swapaxes(b, 1, 2), dt).transpose(1, 2) if b_t else up(b, dt)
    check(down(R.matmul(up(a, dt), bd)), a, b, dt)


@pytest.mark.parametrize("dt", ["f32", "bf16", "f16"])
@pytest.mark.parametrize("a_t,b_t", [(0, 0), (0, 1), (1, 0), (1, 1)])
@pytest.mark.parametrize("batch,m,n", [(3, 70, 61), (130, 255, 241)])
@pytest.mark.parametrize("k", [4, 9, 32, 40, 41, 63, 64, 65, 80, 95, 96, 97, 128, 129, 160, 161, 193])
def test_every_length_of_k_that_changes_the_form(R, dt, a_t, b_t, batch, m, n, k):
    """K up to each size of a single stage (64, 96 and 128 of 16 bits, 32, 48 and 64 of f32) and beyond, in two stages; a few tiles and
    three thousand; what lies around the operands is NaN."""
    g = np.random.Generator(np.random.PCG64(k))
    a, b = rand(g, (3, m, k), dt), rand(g, (3, k, n), dt)
    pad = lambda x: np.pad(x, ((0, 0), (1, 1), (3, 3)), constant_values=np.nan)  # noqa: E731
    some = np.arange(batch) % 3   # the same few products over and over: the batch's strides are checked, the oracle stays small
    A, B = pad(np.swapaxes(a, 1, 2) if a_t else a)[some], pad(np.swapaxes(b, 1, 2) if b_t else b)[some]
    ad = up(A, dt).narrow(1, 1, A.shape[1] - 2).narrow(2, 3, A.shape[2] - 6)
    bd = up(B, dt).narrow(1, 1, B.shape[1] - 2).narrow(2, 3, B.shape[2] - 6)
    got = down(R.matmul(ad.transpose(1, 2) if a_t else ad, bd.transpose(1, 2) if b_t else bd))
    check(got[:3], a, b, dt)
    assert all(np.array_equal(got[i], got[i % 3]) for i in range(3, batch))


@pytest.mark.parametrize("dt", ["f32", "bf16", "f16"])
@pytest.mark.parametrize("a_t,b_t", [(0, 0), (0, 1), (1, 0), (1, 1)])
@pytest.mark.parametrize("m,k,n", [(5, 3, 70), (3, 300, 5), (70, 200, 7), (2, 2, 2), (67, 130, 66)])
def test_operands_of_less_than_a_piece(R, dt, a_t, b_t, m, k, n):
    test_layouts_and_tile_edges(R, dt, a_t, b_t, 2, m, k, n)


@pytest.mark.parametrize("dt", ["f32", "bf16", "f16"])
def test_views_broadcasts_and_general_strides(R, dt):
    g = np.random.Generator(np.random.PCG64(7))
    # heads of a [B, S, H, D] tensor, first feature dropped: strided batches, rows off any alignment
    q, kv = rand(g, (2, 19, 3, 41), dt), rand(g, (2, 23, 3, 41), dt)
    qd, kd = up(q, dt).transpose(1, 2).narrow(3, 1, 40), up(kv, dt).transpose(1, 2).narrow(3, 1, 40)
    qs, ks = np.swapaxes(q, 1, 2)[..., 1:], np.swapaxes(kv, 1, 2)[..., 1:]
    check(down(R.matmul(qd, kd.transpose(2, 3))), qs, np.swapaxes(ks, 2, 3), dt)
    # one operand shared by the batch, on either side; a row and a column broadcast into matrices
    a, b = rand(g, (1, 30, 50), dt), rand(g, (4, 50, 20), dt)
    check(down(R.matmul(up(a, dt), up(b, dt))), a, b, dt)
    check(down(R.matmul(up(b, dt).transpose(1, 2), up(a, dt).transpose(1, 2))), np.swapaxes(b, 1, 2), np.swapaxes(a, 1, 2), dt)
    row, col = rand(g, (3, 1, 50), dt), rand(g, (3, 30, 1), dt)
    rows, cols = np.broadcast_to(row, (3, 30, 50)), np.broadcast_to(col, (3, 30, 50))
    w = rand(g, (3, 50, 9), dt)
    check(down(R.matmul(up(row, dt).broadcast_to((3, 30, 50)), up(w, dt))), rows, w, dt)
    check(down(R.matmul(up(col, dt).broadcast_to((3, 30, 50)), up(w, dt))), cols, w, dt)
    # no unit stride on either axis: the general kernel
    x = rand(g, (2, 12, 3, 14, 2), dt)
    xd = up(x, dt).permute((0, 2, 1, 3, 4)).narrow(4, 0, 1)
    xd = type(xd)(xd.buf, xd.dtype, xd.shape[:4], xd.strides[:4], xd.offset)
    xs = np.transpose(x, (0, 2, 1, 3, 4))[..., 0]
    check(down(R.matmul(xd, xd.transpose(2, 3))), xs, np.swapaxes(xs, 2, 3), dt)


@pytest.mark.parametrize("dt,small", [("f32", 2.0 ** -140), ("bf16", 2.0 ** -130), ("f16", 2.0 ** -22)])
def test_small_and_infinite_values(R, dt, small):
    """Subnormal inputs count, and an infinity or a NaN reaches only the outputs that depend on it (zeros stand past the
    ends of K and of the rows)."""
    for k in (50, 300):
        a, b = np.full((2, 9, k), small, np.float32), np.full((2, k, 11), 2.0 ** 10, np.float32)
        check(down(R.matmul(up(a, dt), up(b, dt))), a, b, dt)
        a, b = np.ones((2, 9, k), np.float32), np.ones((2, k, 11), np.float32)
        a[1, 8, k - 1], b[0, k - 1, 10], b[1, 0, 0] = np.inf, np.nan, np.inf
        got, want = down(R.matmul(up(a, dt), up(b, dt))), np.full((2, 9, 11), k, np.float32)
        want[0, :, 10], want[1, 8], want[1, :, 0] = np.nan, np.inf, np.inf
        np.testing.assert_array_equal(got, want)

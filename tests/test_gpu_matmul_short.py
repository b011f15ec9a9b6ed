"""Batched products A B^T of 16-bit operands in whole 16-byte pieces along a K of up to 128: every number of pieces, both tile sizes, tiles that end past M
and N, batches that stand still, rows with a gap behind them; and infinities, which zeros past K must not meet."""
import numpy as np
import pytest

from tests.util import down, rand, up

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def R(hip):
    from rai_amd import ops

    return ops


def check(R, a, b, dt, ta=None, tb=None):
    ta, tb = ta or up(a, dt), tb or up(b, dt)
    got = down(R.matmul(ta, tb.transpose(1, 2))).astype(np.float64)
    a, b = a.astype(np.float64), b.astype(np.float64).transpose(0, 2, 1)
    want, size = a @ b, np.abs(a) @ np.abs(b)
    # one rounding to the type, and any order of K f32 additions
    assert np.all(np.abs(got - want) <= {"bf16": 2.0 ** -8, "f16": 2.0 ** -11}[dt] * np.abs(want) + (a.shape[2] + 8) * 2.0 ** -24 * size + 2.0 ** -25)


@pytest.mark.parametrize("dt", ["bf16", "f16"])
@pytest.mark.parametrize("k", list(range(8, 136, 8)))
@pytest.mark.parametrize("batch,m,n", [(2, 65, 70), (33, 257, 385)])   # 64 x 64 tiles, 128 x 128
def test_pieces_of_k(R, dt, k, batch, m, n):
    g = np.random.Generator(np.random.PCG64(k + batch))
    check(R, rand(g, (batch, m, k), dt), rand(g, (batch, n, k), dt), dt)


@pytest.mark.parametrize("m,n", [(1, 1), (1, 777), (129, 1), (128, 128), (127, 9), (130, 263), (64, 200)])
def test_ends(R, m, n):
    g = np.random.Generator(np.random.PCG64(m * 1000 + n))
    check(R, rand(g, (40, m, 72), "bf16"), rand(g, (40, n, 72), "bf16"), "bf16")


def test_gap_behind_rows_and_infinities(R):
    g = np.random.Generator(np.random.PCG64(7))
    a, b = rand(g, (3, 70, 64), "bf16"), rand(g, (3, 90, 64), "bf16")
    a[:, :, 24:] = np.inf   # lies behind the K of the view below
    b[:, :, 24:] = np.nan
    check(R, a[:, :, :24], b[:, :, :24], "bf16", up(a, "bf16").narrow(2, 0, 24), up(b, "bf16").narrow(2, 0, 24))


@pytest.mark.parametrize("m,n", [(70, 130), (600, 520)])
def test_one_left_operand_for_every_batch(R, m, n):
    g = np.random.Generator(np.random.PCG64(m))
    a, b = rand(g, (1, m, 40), "f16"), rand(g, (12, n, 40), "f16")
    check(R, np.broadcast_to(a, (12, m, 40)), b, "f16", up(a, "f16"), up(b, "f16"))

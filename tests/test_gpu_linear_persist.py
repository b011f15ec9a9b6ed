"""bf16 Linears on the 256 x 256 tiles of one block per CU (csrc/gemm_persist.hip): one to seven K stages, fewer tiles than CUs
and up to three a block, ragged edges, and every way its outputs leave: bias and activation, gated pairs, residual, two outputs,
rows off 16- and 64-byte boundaries, and what goes row by row (bias and residual, f32 results)."""
import numpy as np
import pytest

from tests.util import down, rand, up

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def R(hip):
    from rai_amd import ops

    return ops


@pytest.fixture(autouse=True)
def forced(monkeypatch):
    monkeypatch.setenv("RAI_HIP_GEMM_TILE", "256x256x8wk64")   # whole 256 x 256 tiles, K never cut


def case(m, k, n):
    g = np.random.Generator(np.random.PCG64(m * 1000 + k + n))
    x, w = rand(g, (m, k), "bf16"), rand(g, (n, k), "bf16", k ** -0.5)
    want = x @ w.T   # in f32: both sides' sums are within the spread of the exact ones
    # any order of K f32 additions and of the bias, twice
    tol = 2 * (k + 20) * 2.0 ** -24 * (np.abs(x) @ np.abs(w).T + 1)
    return x, w, rand(g, (n,), "bf16"), rand(g, (m, n), "bf16"), want, tol


def near(got, want, tol):
    assert np.all(np.abs(got.astype(np.float64) - want) <= 2.0 ** -8 * np.abs(want) + tol)


def silu(z):
    return z / (1 + np.exp(-z))


# tiles: 1, 1 (ragged), 4, 4, 9, 260 (two a block on four CUs), 323, 600 (three a block)
SIZES = [(256, 64, 256), (65, 128, 8), (257, 64, 264), (300, 192, 520), (513, 448, 520), (3328, 64, 5120), (4353, 128, 4872), (5120, 64, 7680)]


@pytest.mark.parametrize("m,k,n", SIZES)
def test_outputs(R, m, k, n):
    x, w, b, r, want, tol = case(m, k, n)
    xd, wd, bd, rd = up(x, "bf16"), up(w, "bf16"), up(b, "bf16"), up(r, "bf16")
    near(down(R.linear(xd, wd)), want, tol)
    near(down(R.linear(xd, wd, residual=rd)), want + r, tol)
    z = want + b
    near(down(R.linear(xd, wd, bd, "silu")), silu(z), 2 * tol + 2.0 ** -18 * np.abs(z) + 2.0 ** -20)   # silu's slope < 1.1, its own error below 2^-18
    near(down(R.linear(xd, wd, bd, "silu", rd)), silu(z) + r, 2 * tol + 2.0 ** -18 * np.abs(z) + 2.0 ** -20)


@pytest.mark.parametrize("m,k,n", [(300, 128, 528), (3328, 64, 5120), (300, 128, 520)])
def test_gated(R, m, k, n):
    x, w, _, _, want, tol = case(m, k, n)
    g, u = want[:, 0::2], want[:, 1::2]
    a = silu(g)
    # gate, up and activation each rounded once (2^-9) before the product, and the product: 2^-8 covers one of the four
    slack = 4 * 2.0 ** -9 * np.abs(a * u) + 2.0 ** -8 * 1.1 * np.abs(g * u) + 2 * (tol[:, 0::2] * (np.abs(u) + 1) + tol[:, 1::2] * (np.abs(a) + 1))
    near(down(R.linear_packed(up(x, "bf16"), up(w, "bf16"), act="silu", glu=True)), a * u, slack)


@pytest.mark.parametrize("n1", [320, 328, 321])
def test_two_outputs(R, n1):
    """The second from a wave's edge, between two, and at an odd column."""
    m, k, n = 300, 192, 712
    x, w, b, _, want, tol = case(m, k, n)
    o1, o2 = R.linear_packed(up(x, "bf16"), up(w, "bf16"), bias=up(b, "bf16"), act="silu", act_from=n1, n1=n1)
    z = want + b
    near(down(o1), z[:, :n1], tol[:, :n1])
    near(down(o2), silu(z[:, n1:]), (2 * tol + 2.0 ** -18 * np.abs(z) + 2.0 ** -20)[:, n1:])


def test_same_bits_whatever_way_the_rows_leave(R):
    """One row of outputs more or fewer to a row moves the rows on other boundaries; the values are the same."""
    m, k = 300, 192
    x, w, _, _, _, _ = case(m, k, 576)
    xd = up(x, "bf16")
    full = down(R.linear(xd, up(w, "bf16")))
    for n in (575, 572, 568, 544):   # 16-byte pieces from the third on, whole 64-byte ones at the last
        np.testing.assert_array_equal(down(R.linear(xd, up(w[:n], "bf16"))), full[:, :n])


# Stream-K: tiles that two and three blocks share (156 tiles), that two share besides a whole round (324), shares before whole tiles (720).
# What the outputs need besides the sums is asked for once these are in.
SHARED = [(3000, 2560, 3104), (4400, 320, 4608), (5000, 256, 9008)]


@pytest.mark.parametrize("m,k,n", SHARED)
def test_outputs_of_shared_tiles(R, monkeypatch, m, k, n):
    monkeypatch.setenv("RAI_HIP_GEMM_TILE", "streamk64")
    test_outputs(R, m, k, n)


@pytest.mark.parametrize("m,k,n", SHARED)
def test_gated_outputs_of_shared_tiles(R, monkeypatch, m, k, n):
    monkeypatch.setenv("RAI_HIP_GEMM_TILE", "streamk64")
    test_gated(R, m, k, n)


@pytest.mark.parametrize("m,k,n", SHARED)
def test_two_outputs_of_shared_tiles_and_the_same_bits_again(R, monkeypatch, m, k, n):
    monkeypatch.setenv("RAI_HIP_GEMM_TILE", "streamk64")
    x, w, b, r, want, tol = case(m, k, n)
    xd, wd, bd, rd = up(x, "bf16"), up(w, "bf16"), up(b, "bf16"), up(r, "bf16")
    n1, z = 1344, want + b
    split = lambda: [down(o) for o in R.linear_packed(xd, wd, bias=bd, act="silu", act_from=n1, n1=n1)]  # noqa: E731
    o1, o2 = split()
    near(o1, z[:, :n1], tol[:, :n1])
    near(o2, silu(z[:, n1:]), (2 * tol + 2.0 ** -18 * np.abs(z) + 2.0 ** -20)[:, n1:])
    added = down(R.linear(xd, wd, residual=rd))
    for _ in range(2):
        again = split()
        assert np.array_equal(again[0], o1) and np.array_equal(again[1], o2)
        assert np.array_equal(down(R.linear(xd, wd, residual=rd)), added)

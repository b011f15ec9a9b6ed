"""bf16 Linears of one to eight rows, at the edges of the kernels that share them out: K around the 512 of a wave's step and
the quarters of a block, odd N, gated pairs, residuals."""
import numpy as np
import pytest

from tests.util import down, rand, up

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def R(hip):
    from rai_amd import ops

    return ops


def spread(x, w):
    """K + 8 roundings of the absolute sum: any order of K f32 additions and the bias."""
    return (x.shape[1] + 8) * 2.0 ** -24 * (np.abs(x.astype(np.float64)) @ np.abs(w.astype(np.float64)).T + 1)


@pytest.mark.parametrize("m", [1, 2, 3, 4, 5, 6, 8])
@pytest.mark.parametrize("k,n", [(8, 1), (8, 5), (504, 2), (520, 1031), (1024, 2049), (2048, 1026), (2056, 3), (4104, 4098), (4096, 8198), (4104, 8193), (8968, 33)])
def test_few_rows(R, m, k, n):
    g = np.random.Generator(np.random.PCG64(m * 1000 + k))
    x, w = rand(g, (m, k), "bf16"), rand(g, (n, k), "bf16", k ** -0.5)
    b, r = rand(g, (n,), "bf16"), rand(g, (m, n), "bf16")
    want = x.astype(np.float64) @ w.astype(np.float64).T
    got = down(R.linear(up(x, "bf16"), up(w, "bf16"))).astype(np.float64)
    assert np.all(np.abs(got - want) <= 2.0 ** -8 * np.abs(want) + spread(x, w))
    z = want + b
    full = z / (1 + np.exp(-z)) + r   # silu's slope stays below 1.1
    got = down(R.linear(up(x, "bf16"), up(w, "bf16"), up(b, "bf16"), "silu", up(r, "bf16"))).astype(np.float64)
    assert np.all(np.abs(got - full) <= 2.0 ** -8 * np.abs(full) + 2 * spread(x, w) + 2.0 ** -20)


@pytest.mark.parametrize("m", [1, 2, 4, 7])
@pytest.mark.parametrize("k,n", [(520, 6), (2560, 1032), (4608, 4112)])
def test_few_rows_gated(R, m, k, n):
    """act(gate) * up with gate, act(gate) and up each rounded to bf16: three roundings, and the sums' own error through a
    product of factors below 8 in size."""
    g = np.random.Generator(np.random.PCG64(m + n))
    x, w = rand(g, (m, k), "bf16"), rand(g, (n, k), "bf16", k ** -0.5)
    z = x.astype(np.float64) @ w.astype(np.float64).T
    gate, upv = z[:, 0::2], z[:, 1::2]
    want = gate / (1 + np.exp(-gate)) * upv
    got = down(R.linear_packed(up(x, "bf16"), up(w, "bf16"), act="silu", glu=True)).astype(np.float64)
    size = (np.abs(gate) + 1) * (np.abs(upv) + 1)
    assert np.all(np.abs(got - want) <= 4 * 2.0 ** -8 * size)


@pytest.mark.parametrize("m", [1, 2, 3, 5, 8])
@pytest.mark.parametrize("k,n,n1", [(520, 39, 17), (2560, 1031, 301), (4104, 8200, 4099), (8968, 40, 8)])
def test_few_rows_two_outputs(R, m, k, n, n1):
    """Columns [0, n1) without, the rest with an activation, into a second output; n1 odd: rows of no alignment."""
    g = np.random.Generator(np.random.PCG64(m * 1000 + k))
    x, w, b = rand(g, (m, k), "bf16"), rand(g, (n, k), "bf16", k ** -0.5), rand(g, (n,), "bf16")
    z = x.astype(np.float64) @ w.astype(np.float64).T + b
    want = np.concatenate([z[:, :n1], z[:, n1:] / (1 + np.exp(-z[:, n1:]))], 1)
    o1, o2 = R.linear_packed(up(x, "bf16"), up(w, "bf16"), bias=up(b, "bf16"), act="silu", act_from=n1, n1=n1)
    assert o1.shape == (m, n1) and o2.shape == (m, n - n1)
    got = np.concatenate([down(o1), down(o2)], 1).astype(np.float64)
    assert np.all(np.abs(got - want) <= 2.0 ** -8 * np.abs(want) + 2 * spread(x, w) + 2.0 ** -20)   # silu's slope stays below 1.1


@pytest.mark.parametrize("m", [1, 2, 4, 6, 7])
@pytest.mark.parametrize("k,n", [(504, 5), (2048, 2050), (4608, 8195)])
def test_few_rows_two_biases(R, m, k, n):
    """The activation from a column on within one output, two biases, a residual."""
    g = np.random.Generator(np.random.PCG64(m + n))
    x, w, r = rand(g, (m, k), "bf16"), rand(g, (n, k), "bf16", k ** -0.5), rand(g, (m, n), "bf16")
    b, b2 = rand(g, (n,), "bf16"), rand(g, (n,), "bf16")
    z = x.astype(np.float64) @ w.astype(np.float64).T + (b.astype(np.float64) + b2)
    at = n // 2
    z[:, at:] = z[:, at:] / (1 + np.exp(-z[:, at:]))
    want = z + r
    got = down(R.linear_packed(up(x, "bf16"), up(w, "bf16"), bias=up(b, "bf16"), bias2=up(b2, "bf16"), act="silu", act_from=at, residual=up(r, "bf16")))
    # the three additions after the sum: a rounding each of what they add
    extra = 2.0 ** -23 * (np.abs(b) + np.abs(b2) + np.abs(z) + np.abs(r))
    assert np.all(np.abs(got.astype(np.float64) - want) <= 2.0 ** -8 * np.abs(want) + 2 * spread(x, w) + extra + 2.0 ** -20)


@pytest.mark.parametrize("m,n", [(9, 68), (31, 132)])
@pytest.mark.parametrize("splits", [2, 3, 5, 7, 8, 9, 13])
def test_parts_of_k_by_batches(R, monkeypatch, splits, m, n):
    """Nine rows and more with K cut over blocks: the last block reads the parts eight, four, two, one at a time, with the residual
    beside them; the bits of the separate summing pass."""
    k = 2048 * (splits - 1) + 224
    g = np.random.Generator(np.random.PCG64(m + splits))
    x, w = rand(g, (m, k), "bf16"), rand(g, (n, k), "bf16", k ** -0.5)
    b, r = rand(g, (n,), "bf16"), rand(g, (m, n), "bf16")
    args = up(x, "bf16"), up(w, "bf16"), up(b, "bf16"), None, up(r, "bf16")
    got = down(R.linear(*args))
    monkeypatch.setenv("RAI_HIP_NO_FUSED_SPLITK", "1")
    np.testing.assert_array_equal(got, down(R.linear(*args)))
    full = x.astype(np.float64) @ w.astype(np.float64).T + b + r
    assert np.all(np.abs(got - full) <= 2.0 ** -8 * np.abs(full) + spread(x, w))

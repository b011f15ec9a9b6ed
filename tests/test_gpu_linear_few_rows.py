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

"""Attention with a block to a query row: keys in rounds of four to a group of 16 lanes, whole, partly filled and nearly empty
ones; every dtype, rows of a part of 16 pieces, of 16 and of several times 16."""
import numpy as np
import pytest

from tests.test_gpu_attention_f32 import R, reference  # noqa: F401
from tests.util import down, rand, up

pytestmark = pytest.mark.gpu
EPS = {"f32": 2.0 ** -24, "bf16": 2.0 ** -8, "f16": 2.0 ** -11}


@pytest.mark.parametrize("dt", ["f32", "bf16", "f16"])
@pytest.mark.parametrize("d", [8, 40, 48, 96, 136, 256, 320])
@pytest.mark.parametrize("s,t,causal", [(1, 1, 1), (3, 15, 0), (2, 17, 1), (5, 48, 0), (3, 49, 1), (2, 63, 1), (1, 64, 0), (4, 66, 1), (2, 129, 0), (3, 333, 1)])
def test_against_64_bits(R, dt, d, s, t, causal):  # noqa: F811
    g = np.random.Generator(np.random.PCG64(t + d))
    q, k, v = rand(g, (2, 4, s, d), dt), rand(g, (2, 2, t, d), dt), rand(g, (2, 2, t, d), dt)
    want, tol = reference(q, k, v, d ** -0.5, causal)
    weights, _ = reference(q, k, np.abs(v), d ** -0.5, causal)
    # a probability is rounded to the dtype before the product with V, and the result
    tol = tol + EPS[dt] * weights * (1 + EPS[dt]) + EPS[dt] * np.abs(want) + 2.0 ** -24
    got = down(R.attention(up(q, dt), up(k, dt), up(v, dt), d ** -0.5, causal, 1)).astype(np.float64)
    assert np.all(np.abs(got - want) <= tol)

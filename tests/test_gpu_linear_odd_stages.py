"""bf16 Linears whose K is an odd number of 32s: the first stage of 64 begins half a stage before the rows do.  What lies around the
rows is NaN, so that nothing of it may take part; every tile size, K in one part and in several, and the sizes on either side of
the lines between stages of 64 and of 32."""
import numpy as np
import pytest

from tests.test_gpu_linear_persist import R, near, silu  # noqa: F401
from tests.util import down, rand, up

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("m,k,n", [(65, 32, 72), (65, 96, 72), (130, 96, 600), (277, 1376, 600), (70, 2592, 264), (257, 352, 1000), (1024, 2080, 2048), (600, 160, 11000),
                                   (333, 1568, 2960), (777, 288, 3000), (513, 800, 7000), (1300, 416, 8000), (2000, 96, 2000), (2000, 96, 1700), (1900, 800, 2304),
                                   (2100, 800, 4104)])
def test_nothing_before_the_rows(R, m, k, n):  # noqa: F811
    g = np.random.Generator(np.random.PCG64(m + k + n))
    x, w, b, r = rand(g, (m, k), "bf16"), rand(g, (n, k), "bf16", k ** -0.5), rand(g, (n,), "bf16"), rand(g, (m, n), "bf16")
    want = x @ w.T   # in f32, as below any order of K f32 additions and of the bias, twice
    tol = 2 * (k + 20) * 2.0 ** -24 * (np.abs(x) @ np.abs(w).T + 1)
    around = lambda a: np.pad(a, ((0, 0), (64, 40)), constant_values=np.nan)  # noqa: E731
    xd, wd = up(around(x), "bf16").narrow(1, 64, k), up(around(w), "bf16").narrow(1, 64, k)
    near(down(R.linear(xd, wd)), want, tol)
    near(down(R.linear(up(x, "bf16"), up(w, "bf16"), residual=up(r, "bf16"))), want + r, tol)
    z = want + b
    near(down(R.linear(xd, wd, up(b, "bf16"), "silu")), silu(z), 2 * tol + 2.0 ** -18 * np.abs(z) + 2.0 ** -20)


@pytest.mark.parametrize("k", [96, 160, 608])
def test_more_parts_than_stages(R, k):  # noqa: F811
    """The first part always has a second stage: what it asks for again past its last one would begin before the rows."""
    g = np.random.Generator(np.random.PCG64(k))
    x, w = rand(g, (130, k), "bf16"), rand(g, (264, k), "bf16", k ** -0.5)
    tol = 2 * (k + 20) * 2.0 ** -24 * (np.abs(x) @ np.abs(w).T + 1)
    for parts in (1, 2, 3, 5, 9, 40):
        near(down(R.linear_packed(up(x, "bf16"), up(w, "bf16"), k_splits=parts)), x @ w.T, tol)

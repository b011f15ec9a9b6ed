"""Norms and softmax of rows that are no whole number of 16-byte pieces: around the lengths where an item more goes to a lane or a thread, on
both sides of the row counts where a wave takes a row, with rows that lie apart by an odd stride or start off a piece."""
import numpy as np
import pytest

from tests.util import down, rand, up

pytestmark = pytest.mark.gpu
U = {"f32": 2.0 ** -24, "bf16": 2.0 ** -8, "f16": 2.0 ** -11}
SIZES = [(1, 1), (3, 63), (4, 65), (5, 129), (2, 255), (3, 257), (7, 511), (4, 513), (1, 1025), (3, 2049), (2, 4095), (3, 4097), (1, 3381),
         (2048, 255), (2049, 63), (2049, 127), (2051, 255), (2050, 257), (8195, 66)]


def views(rows, n, dt):
    """x and the same numbers inside wider rows, from the second element on."""
    g = np.random.Generator(np.random.PCG64(rows * 5 + n))
    x = rand(g, (rows, n + 3), dt, 2.0)
    wide = up(x, dt)
    return [(np.ascontiguousarray(x[:, 1:n + 1]), wide.narrow(1, 1, n)), (np.ascontiguousarray(x[:, :n]), up(np.ascontiguousarray(x[:, :n]), dt))]


@pytest.mark.parametrize("rows,n", SIZES)
@pytest.mark.parametrize("dt", ["f32", "bf16", "f16"])
def test_norms(hip, dt, rows, n):
    from rai_amd import ops as R

    g = np.random.Generator(np.random.PCG64(rows + n))
    w, b = rand(g, (n,), dt), rand(g, (n,), dt)
    for x, xd in views(rows, n, dt):
        d = x.astype(np.float64)

        def check(got, mean, scale, w, b):
            y = (d - mean) * scale
            want = y * w + b
            # sums within n + 8 roundings of n (terms of one sign, or below 2 in the mean), halved by the root; a handful of roundings of
            # the factors; the difference of a value and the mean, in one of a few elements little of either; the result's own
            tol = (n + 16) * 2.0 ** -24 * (np.abs(y) + np.abs(scale) * 4 + 2) * np.abs(w) + 4 * 2.0 ** -24 * np.abs(b) + 2 * U[dt] * np.abs(want) + 2.0 ** -24
            assert np.all(np.abs(down(got).astype(np.float64) - want) <= tol)

        ms = (d * d).mean(-1, keepdims=True)
        check(R.rms_norm(xd, up(w, dt), 1e-2), 0.0, 1 / np.sqrt(ms + 1e-2), w, 0.0)
        check(R.rms_norm(xd, up(w, dt), 1e-2, True), 0.0, 1 / np.sqrt(ms + 1e-2), 1.0 + w, 0.0)
        mean, var = d.mean(-1, keepdims=True), d.var(-1, keepdims=True)
        check(R.layer_norm(xd, up(w, dt), up(b, dt), 1e-2), mean, 1 / np.sqrt(var + 1e-2), w, b)
        check(R.layer_norm(xd, None, None, 1e-2), mean, 1 / np.sqrt(var + 1e-2), 1.0, 0.0)


@pytest.mark.parametrize("rows,n", SIZES)
@pytest.mark.parametrize("dt", ["f32", "bf16", "f16"])
def test_softmax(hip, dt, rows, n):
    from rai_amd import ops as R

    for x, xd in views(rows, n, dt):
        d = x.astype(np.float64)
        d -= d.max(-1, keepdims=True)
        e = np.exp(d)
        y = e / e.sum(-1, keepdims=True)
        # the difference and the exponential within a few roundings (those of the difference grow with it), the sum within n + 8; the result's own
        rel = (n + 16 + 2 * np.abs(d)) * 2.0 ** -24
        assert np.all(np.abs(down(R.softmax(xd, -1)).astype(np.float64) - y) <= rel * y + 2 * U[dt] * y + (2.0 ** -24 if dt == "f16" else 1e-37))
        want = d - np.log(e.sum(-1, keepdims=True))
        assert np.all(np.abs(down(R.log_softmax(xd, -1)).astype(np.float64) - want) <= (n + 16) * 2.0 ** -24 + 4 * 2.0 ** -24 * np.abs(d) + 2 * U[dt] * np.abs(want))


@pytest.mark.parametrize("n", [65, 511, 2049, 4095])
def test_softmax_of_masked_rows(hip, n):
    """Minus infinity has probability zero; a row of nothing else is NaN."""
    from rai_amd import ops as R

    x = np.zeros((5, n), np.float32)
    x[1, 1:] = -np.inf
    x[2] = -np.inf
    x[3, : n // 2] = -np.inf
    got = down(R.softmax(up(x, "f32"), -1))
    assert got[1, 0] == 1.0 and not got[1, 1:].any() and np.isnan(got[2]).all()
    assert not got[3, : n // 2].any() and np.allclose(got[3, n // 2:], 1.0 / (n - n // 2), rtol=(n + 16) * 2.0 ** -24)

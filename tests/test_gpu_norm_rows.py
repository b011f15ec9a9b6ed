"""Norms around the sizes where a row goes from a block to a wave and a thread from one 16-byte piece to the next."""
import numpy as np
import pytest

from tests.util import down, rand, up

pytestmark = pytest.mark.gpu
U = {"f32": 2.0 ** -24, "bf16": 2.0 ** -8, "f16": 2.0 ** -11}


# Columns by 16-byte pieces of 16-bit elements: a wave's two, five and nine pieces a lane at both ends, a block's one to four a thread; rows on
# both sides of 1536, 2048, 4096 and 6144, beyond which the other form may serve.
@pytest.mark.parametrize("rows,n", [(1, 8), (3, 1016), (2, 2048), (5, 2056), (1, 4104), (2, 8192), (1536, 264), (1537, 264), (2048, 264), (2049, 264),
                                    (2049, 1024), (2049, 1032), (2049, 1536), (2051, 1544), (2050, 2048), (4096, 1800), (4097, 1800), (2049, 2304),
                                    (2049, 2312), (6144, 2304), (6145, 2304), (2049, 2560), (2049, 2568), (2049, 3072), (2050, 3080), (2050, 4104),
                                    (2050, 4608), (2050, 4616)])
@pytest.mark.parametrize("dt", ["f32", "bf16", "f16"])
def test_rows(hip, dt, rows, n):
    from rai_amd import ops as R

    if dt == "f32":
        n //= 2   # the same number of 16-byte pieces
    g = np.random.Generator(np.random.PCG64(rows + n))
    x, w, b = rand(g, (rows, n), dt, 2.0), rand(g, (n,), dt), rand(g, (n,), dt)
    d = x.astype(np.float64)

    def check(got, mean, scale, w, b):
        y = (d - mean) * scale
        want = y * w + b
        # the statistics' sums are within n + 8 roundings of n (terms of one sign, or below 2 in the mean), halved by the root; a
        # handful of roundings of the factors; the result's own
        tol = (n + 16) * 2.0 ** -24 * (np.abs(y) + 2) * np.abs(w) + 4 * 2.0 ** -24 * np.abs(b) + 2 * U[dt] * np.abs(want) + 2.0 ** -24
        assert np.all(np.abs(down(got).astype(np.float64) - want) <= tol)

    ms = (d * d).mean(-1, keepdims=True)
    check(R.rms_norm(up(x, dt), up(w, dt), 1e-6), 0.0, 1 / np.sqrt(ms + 1e-6), w, 0.0)
    check(R.rms_norm(up(x, dt), up(w, dt), 1e-6, True), 0.0, 1 / np.sqrt(ms + 1e-6), 1.0 + w, 0.0)
    mean, var = d.mean(-1, keepdims=True), d.var(-1, keepdims=True)
    check(R.layer_norm(up(x, dt), up(w, dt), up(b, dt), 1e-5), mean, 1 / np.sqrt(var + 1e-5), w, b)
    check(R.layer_norm(up(x, dt), None, None, 1e-5), mean, 1 / np.sqrt(var + 1e-5), 1.0, 0.0)


@pytest.mark.parametrize("dt,n", [("f32", 4), ("f32", 1028), ("bf16", 1544)])
def test_more_rows_than_one_grid_dimension_holds(hip, dt, n):
    """2^24 rows and a few: 2^32 threads where a block of 256 has a row.  Equal rows, read with a stride of zero; the output (up to
    69 GB) is looked at around every power of two that a count of rows or threads could be cut off at."""
    from rai_amd import ops as R
    from rai_amd._lib import call

    rows = (1 << 24) + 5
    g = np.random.Generator(np.random.PCG64(n))
    x, w, b = rand(g, (n,), dt, 2.0), rand(g, (n,), dt), rand(g, (n,), dt)
    many = up(x, dt).broadcast_to((rows, n))
    for fn in (lambda t: R.rms_norm(t, up(w, dt), 1e-6), lambda t: R.layer_norm(t, up(w, dt), up(b, dt), 1e-5)):
        want, got = down(fn(up(x[None], dt))), fn(many)
        for at in (0, (1 << 22) - 2, (1 << 23) - 2, (1 << 24) - 2, rows - 4):
            part = down(got.narrow(0, at, 4)).astype(np.float64)
            # one row and many may be served by different kernels: both are within an f32 norm's roundings and one of dt
            assert np.all(np.abs(part - want) <= (n + 16) * 2.0 ** -23 * (np.abs(want) + 4 * np.abs(w) + np.abs(b)) + 2 * U[dt] * np.abs(want)), at
        del got
        call("rai_hip_trim", 0)

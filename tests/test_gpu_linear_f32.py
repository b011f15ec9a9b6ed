"""f32 Linears at the edges of their kernels' tiles: rows around 4, 32 and 64, K around the 32-wide tiles and the cut over
waves and blocks, odd N, rows that are not 16-byte aligned."""
import threading

import numpy as np
import pytest

from tests.util import down, rand, up

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def R(hip):
    from rai_amd import ops

    return ops


def bound(x, w, extra):
    """Every sum of K products in f32, whatever its order, is within K roundings of the absolute sum; the epilogue's
    few roundings and its activation are within eight of the result's own size and of what was added."""
    return (x.shape[1] + 8) * 2.0 ** -24 * (np.abs(x.astype(np.float64)) @ np.abs(w.astype(np.float64)).T) + 2.0 ** -20 * extra


@pytest.mark.parametrize("m", [1, 2, 3, 4, 5, 31, 33, 64, 65, 130])
@pytest.mark.parametrize("k,n", [(4, 1), (36, 70), (33, 129), (252, 64), (260, 63), (1028, 258), (2560, 40)])
def test_f32_linear_at_tile_edges(R, m, k, n):
    g = np.random.Generator(np.random.PCG64(31 + m))
    x, w = rand(g, (m, k), "f32"), rand(g, (n, k), "f32", 0.05)
    b, r = rand(g, (n,), "f32"), rand(g, (m, n), "f32")
    want = x.astype(np.float64) @ w.astype(np.float64).T
    got = down(R.linear(up(x, "f32"), up(w, "f32"))).astype(np.float64)
    assert np.all(np.abs(got - want) <= bound(x, w, 0.0))
    z = want + b
    full = 0.5 * z * (1 + np.tanh(np.sqrt(2 / np.pi) * (z + 0.044715 * z ** 3))) + r
    got = down(R.linear(up(x, "f32"), up(w, "f32"), up(b, "f32"), "new_gelu", up(r, "f32"))).astype(np.float64)
    assert np.all(np.abs(got - full) <= 2 * bound(x, w, np.abs(z) + np.abs(r) + 1))   # the activation's slope is below 1.13


@pytest.mark.parametrize("m", [1, 3, 40])
def test_f32_linear_of_unaligned_rows(R, m):
    """A weight matrix and activations that start one element into their buffers, rows an odd number of elements apart."""
    g = np.random.Generator(np.random.PCG64(77))
    x, w = rand(g, (m, 133), "f32"), rand(g, (50, 131), "f32", 0.05)
    got = down(R.linear(up(x, "f32").narrow(1, 1, 128), up(w, "f32").narrow(1, 3, 128))).astype(np.float64)
    xs, ws = x[:, 1:129], w[:, 3:131]
    assert np.all(np.abs(got - xs.astype(np.float64) @ ws.astype(np.float64).T) <= bound(xs, ws, 0.0))


@pytest.mark.parametrize("m,n", [(2, 9), (70, 66), (64, 1600)])
@pytest.mark.parametrize("k", [1, 2, 3, 5, 6, 7, 30, 31, 35, 66, 511, 1026])
def test_f32_linear_where_k_ends_inside_a_piece(R, m, n, k):
    """K of no multiple of four, rows packed, on 16-byte boundaries and off them; what stands behind a row's end, and the
    first elements of the next row, take no part."""
    g = np.random.Generator(np.random.PCG64(13))
    for first, width in ((0, k), (0, (k + 3) // 4 * 4 + 4), (1, k + 3)):
        x, w = rand(g, (m, width), "f32"), rand(g, (n, width), "f32", 0.05)
        x[:, :first] = w[:, :first] = x[:, first + k:] = w[:, first + k:] = np.nan
        got = down(R.linear(up(x, "f32").narrow(1, first, k), up(w, "f32").narrow(1, first, k))).astype(np.float64)
        xs, ws = x[:, first:first + k], w[:, first:first + k]
        assert np.all(np.abs(got - xs.astype(np.float64) @ ws.astype(np.float64).T) <= bound(xs, ws, 0.0)), (first, width)


@pytest.mark.parametrize("m,k,n", [(4, 4096, 512), (32, 4096, 8192)])
def test_unaligned_rows_are_cut_by_the_tiles_they_get(R, m, k, n):
    """Rows off 16-byte boundaries take 64 x 64 tiles however few they are, so as few as these are cut over K like 40: the
    same parts of K, and the same bits."""
    g = np.random.Generator(np.random.PCG64(17))
    x, w = up(rand(g, (40, k + 1), "f32"), "f32").narrow(1, 1, k), up(rand(g, (n, k + 1), "f32", 0.02), "f32").narrow(1, 1, k)
    assert np.array_equal(down(R.linear(x.narrow(0, 0, m), w)), down(R.linear(x, w))[:m])


@pytest.mark.parametrize("m", [1, 2, 3, 4])
@pytest.mark.parametrize("k,n", [(64, 10241), (256, 16385), (512, 16390), (1024, 16390)])
def test_f32_few_rows_against_many_short_weights(R, m, k, n):
    """Both sides of the line between the few-row kernel and the tiles."""
    g = np.random.Generator(np.random.PCG64(19))
    x, w, b, r = rand(g, (m, k), "f32"), rand(g, (n, k), "f32", 0.05), rand(g, (n,), "f32"), rand(g, (m, n), "f32")
    want = x.astype(np.float64) @ w.astype(np.float64).T + b + r
    got = down(R.linear(up(x, "f32"), up(w, "f32"), up(b, "f32"), None, up(r, "f32"))).astype(np.float64)
    assert np.all(np.abs(got - want) <= bound(x, w, np.abs(b) + np.abs(r)))


@pytest.mark.parametrize("m", [1, 20, 100])
def test_f32_linear_keeps_small_and_infinite_values(R, m):
    """Denormal products are kept, and infinities and NaNs reach only the outputs that depend on them (K is no multiple
    of a tile, so zeros stand past its end)."""
    x = np.full((m, 300), np.float32(2.0 ** -70))
    w = np.full((70, 300), np.float32(2.0 ** -65))
    assert np.all(down(R.linear(up(x, "f32"), up(w, "f32"))) == np.float32(300 * 2.0 ** -135))
    x = np.ones((m, 300), np.float32)
    w = np.ones((70, 300), np.float32)
    w[7, 299], w[9, 0] = np.inf, np.nan
    got = down(R.linear(up(x, "f32"), up(w, "f32")))
    assert np.all(np.isinf(got[:, 7])) and np.all(np.isnan(got[:, 9])) and np.all(np.delete(got, [7, 9], 1) == 300)


@pytest.mark.parametrize("dt", ["f32", "bf16"])
@pytest.mark.parametrize("planes", [0, 1, 3])
def test_linear_runs_where_the_scratch_cannot_grow(R, monkeypatch, dt, planes):
    """A product that would cut K needs no memory of its own to run: without room for all its partial sums it runs in
    fewer parts or in one."""
    g = np.random.Generator(np.random.PCG64(78))
    m, k, n = 96, 4096, 520
    x, w = rand(g, (m, k), dt), rand(g, (n, k), dt, 0.02)
    xd, wd = up(x, dt), up(w, dt)
    first = down(R.linear(xd, wd))
    monkeypatch.setenv("RAI_HIP_WORKSPACE_LIMIT", str(planes * m * n * 4))
    got = down(R.linear(xd, wd)).astype(np.float64)
    want = x.astype(np.float64) @ w.astype(np.float64).T
    assert np.all(np.abs(got - want) <= bound(x, w, 0.0) + (2.0 ** -8 * np.abs(want) if dt == "bf16" else 0.0))
    monkeypatch.delenv("RAI_HIP_WORKSPACE_LIMIT")
    assert np.array_equal(down(R.linear(xd, wd)), first)


def test_linears_of_several_threads_share_the_scratch(R):
    """Products that cut K leave partial sums in the device's one scratch block between two kernels: threads that launch
    them at the same time, with sizes that make the block grow on the way, get the bits that each gets alone."""
    sizes = [(48, 4096, 512, "f32"), (96, 4096, 1024, "f32"), (128, 8192, 512, "bf16"), (200, 8192, 2560, "f32")]

    def operands(i):
        m, k, n, dt = sizes[i]
        g = np.random.Generator(np.random.PCG64(91 + i))
        return up(rand(g, (m, k), dt), dt), up(rand(g, (n, k), dt, k ** -0.5), dt)

    data, got = [operands(i) for i in range(len(sizes))], [[] for _ in sizes]

    def work(i):
        got[i] = [R.linear(*data[i]) for _ in range(25)]

    threads = [threading.Thread(target=work, args=(i,)) for i in range(len(sizes))]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    for i, outs in enumerate(got):
        alone = down(R.linear(*data[i]))
        assert len(outs) == 25 and all(np.array_equal(down(y), alone) for y in outs), sizes[i]

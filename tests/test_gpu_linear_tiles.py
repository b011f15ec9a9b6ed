"""bf16 Linears of more than eight rows on tiles with K stages of 64: as the sizes choose them (64 x 64 for most of these; the
rule's pick of every tile, cut over K and whole, is asked for and asserted below), and each tile forced, with one to as many stages
as it keeps in flight and one more, ragged edges, K in parts, gated pairs."""
import ctypes as C

import numpy as np
import pytest

from tests.util import down, rand, up

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def R(hip):
    from rai_amd import ops

    return ops


def spread(x, w):
    """K + 20 roundings of the absolute sum: any order of K f32 additions, of the parts of K and of the bias."""
    return (x.shape[1] + 20) * 2.0 ** -24 * (np.abs(x.astype(np.float64)) @ np.abs(w.astype(np.float64)).T + 1)


SIZES = [(65, 64, 8), (65, 128, 65), (97, 192, 1031), (129, 256, 257), (333, 320, 520), (72, 1536, 512), (100, 2048, 2050), (333, 2048, 72),
         (9, 64, 4096), (16, 192, 4104), (64, 1536, 2048), (40, 2048, 4097), (15, 4096, 2056), (64, 576, 9000),
         (1000, 512, 2048), (530, 1088, 1500), (333, 1088, 8968), (130, 2560, 8200), (600, 1152, 5000), (65, 1664, 512), (65, 1216, 520)]


@pytest.mark.parametrize("m,k,n", SIZES)
def test_tiles(R, m, k, n):
    g = np.random.Generator(np.random.PCG64(m * 1000 + k))
    x, w = rand(g, (m, k), "bf16"), rand(g, (n, k), "bf16", k ** -0.5)
    b, r = rand(g, (n,), "bf16"), rand(g, (m, n), "bf16")
    want, tol = x.astype(np.float64) @ w.astype(np.float64).T, spread(x, w)
    got = down(R.linear(up(x, "bf16"), up(w, "bf16"))).astype(np.float64)
    assert np.all(np.abs(got - want) <= 2.0 ** -8 * np.abs(want) + tol)
    z = want + b
    full = z / (1 + np.exp(-z)) + r   # silu's slope stays below 1.1, its own error below 2^-18 of it
    got = down(R.linear(up(x, "bf16"), up(w, "bf16"), up(b, "bf16"), "silu", up(r, "bf16"))).astype(np.float64)
    assert np.all(np.abs(got - full) <= 2.0 ** -8 * np.abs(full) + 2 * tol + 2.0 ** -18 * np.abs(z) + 2.0 ** -20)


TILES = ["64x64", "128x64", "128x128k64", "128x128deep", "128x256", "192x256", "256x192", "256x256k64"]   # (128x128k64 and 128x128deep: one kernel)


@pytest.mark.parametrize("m,k,n", [(65, 64, 8), (129, 128, 257), (200, 192, 136), (333, 256, 520), (72, 320, 1031), (65, 1664, 512), (260, 1088, 300), (130, 2560, 776)])
@pytest.mark.parametrize("tile", TILES)
def test_every_tile(R, monkeypatch, tile, m, k, n):
    monkeypatch.setenv("RAI_HIP_GEMM_TILE", tile)   # read per call; K is cut as the tile's own plan says
    test_tiles(R, m, k, n)


@pytest.mark.parametrize("m,k,n,parts", [(65, 192, 136, 3), (65, 448, 136, 3), (130, 640, 200, 4), (97, 832, 264, 12)])
@pytest.mark.parametrize("tile", TILES)
def test_parts_shorter_than_the_pipeline(R, monkeypatch, tile, m, k, n, parts):
    """Parts of one, two and three stages of K."""
    monkeypatch.setenv("RAI_HIP_GEMM_TILE", tile)
    g = np.random.Generator(np.random.PCG64(k))
    x, w, b, r = rand(g, (m, k), "bf16"), rand(g, (n, k), "bf16", k ** -0.5), rand(g, (n,), "bf16"), rand(g, (m, n), "bf16")
    want = x.astype(np.float64) @ w.astype(np.float64).T + b + r
    got = down(R.linear_packed(up(x, "bf16"), up(w, "bf16"), bias=up(b, "bf16"), residual=up(r, "bf16"), k_splits=parts)).astype(np.float64)
    assert np.all(np.abs(got - want) <= 2.0 ** -8 * np.abs(want) + 2 * spread(x, w))


@pytest.mark.parametrize("k,parts", [(64, 2), (128, 3), (64, 7)])
def test_more_parts_asked_for_than_k_has_stages(R, k, parts):
    g = np.random.Generator(np.random.PCG64(k))
    x, w = rand(g, (100, k), "bf16"), rand(g, (136, k), "bf16", k ** -0.5)
    want = x.astype(np.float64) @ w.astype(np.float64).T
    down(R.linear_packed(up(-x, "bf16"), up(w, "bf16")))   # (an output that is not written may still hold its like)
    got = down(R.linear_packed(up(x, "bf16"), up(w, "bf16"), k_splits=parts)).astype(np.float64)
    assert np.all(np.abs(got - want) <= 2.0 ** -8 * np.abs(want) + spread(x, w))


@pytest.mark.parametrize("tile", TILES)
def test_every_tile_gated(R, monkeypatch, tile):
    monkeypatch.setenv("RAI_HIP_GEMM_TILE", tile)
    for m, k, n in [(70, 256, 136), (300, 1536, 520)]:
        test_tiles_gated(R, m, k, n)


@pytest.mark.parametrize("m,k,n", [(70, 256, 136), (300, 1536, 520), (20, 1536, 4104), (256, 2048, 2048)])
def test_tiles_gated(R, m, k, n):
    """act(gate) * up with gate, act(gate) and up each rounded to bf16: three roundings, and the sums' own error through a
    product of factors below 8 in size."""
    g = np.random.Generator(np.random.PCG64(m + n))
    x, w = rand(g, (m, k), "bf16"), rand(g, (n, k), "bf16", k ** -0.5)
    z = x.astype(np.float64) @ w.astype(np.float64).T
    gate, upv = z[:, 0::2], z[:, 1::2]
    want = gate / (1 + np.exp(-gate)) * upv
    got = down(R.linear_packed(up(x, "bf16"), up(w, "bf16"), act="silu", glu=True)).astype(np.float64)
    assert np.all(np.abs(got - want) <= 4 * 2.0 ** -8 * (np.abs(gate) + 1) * (np.abs(upv) + 1))


# The eight-wave tiles of 256 columns: short K (stages fewer than the pipeline), ragged rows and columns, parts of K.
@pytest.mark.parametrize("m,k,n", [(65, 64, 8), (129, 128, 257), (193, 192, 520), (383, 256, 1031), (385, 1088, 264), (130, 2560, 776)])
@pytest.mark.parametrize("tile", ["128x256", "192x256", "256x192", "256x256k64"])
def test_wide_tiles(R, monkeypatch, tile, m, k, n):
    monkeypatch.setenv("RAI_HIP_GEMM_TILE", tile)
    test_tiles(R, m, k, n)
    test_tiles_gated(R, m, k, 8 * (n // 8))


def plan(m, k, n):
    """(tile, parts of K) that the rule gives R.linear."""
    from rai_amd._lib import call

    name, parts = C.create_string_buffer(32), C.c_int32()
    call("rai_hip_linear_plan", 0, m, k, n, min(32 * m * n, 256 << 20), name, 32, C.byref(parts))
    return name.value.decode(), parts.value


# What the rule picks by itself: every tile whole and, where it is ever the best, cut over K.
@pytest.mark.parametrize("m,k,n,tile,cut", [
    (87, 320, 312, "64x64", False), (68, 2176, 288, "64x64", True), (675, 192, 5432, "128x64", False), (69, 3840, 3376, "128x64", True),
    (1450, 448, 1552, "128x128k64", False), (65, 5632, 3424, "128x128k64", True), (393, 320, 12728, "128x256", False), (130, 6400, 5560, "128x256", True),
    (3692, 448, 2232, "192x256", False), (259, 3520, 11096, "192x256", True), (4843, 192, 2312, "256x192", False), (8352, 384, 1552, "256x256k64", False),
    (409, 5760, 8416, "256x256k64", True), (4000, 2560, 10200, "streamk64", False)])
def test_what_the_rule_picks(R, m, k, n, tile, cut):
    picked, parts = plan(m, k, n)
    assert (picked, parts > 1) == (tile, cut), (picked, parts)
    g = np.random.Generator(np.random.PCG64(m * 1000 + k))
    x, w, b, r = rand(g, (m, k), "bf16"), rand(g, (n, k), "bf16", k ** -0.5), rand(g, (n,), "bf16"), rand(g, (m, n), "bf16")
    xd, wd = up(x, "bf16"), up(w, "bf16")
    want = x @ w.T   # in f32: both sides' sums are within the spread of the exact ones
    tol = 2 * (k + 20) * 2.0 ** -24 * (np.abs(x) @ np.abs(w).T + 1)
    assert np.all(np.abs(down(R.linear(xd, wd)) - want) <= 2.0 ** -8 * np.abs(want) + tol)
    z = want + b
    full = z / (1 + np.exp(-z)) + r   # silu's slope stays below 1.1, its own error below 2^-18 of it
    got = down(R.linear(xd, wd, up(b, "bf16"), "silu", up(r, "bf16")))
    assert np.all(np.abs(got - full) <= 2.0 ** -8 * np.abs(full) + 2 * tol + 2.0 ** -18 * np.abs(z) + 2.0 ** -20)


@pytest.mark.parametrize("tile", ["256x256k64", "streamk64"])
def test_operands_that_no_cache_holds(R, monkeypatch, tile):
    """290 MB of operands: 256 x 256 tiles of a block each, and their shares; ragged rows, columns and number of stages."""
    monkeypatch.setenv("RAI_HIP_GEMM_TILE", tile)
    m, k, n, few = 16200, 8256, 1400, 300
    g = np.random.Generator(np.random.PCG64(m + k))
    x, w, b, r = rand(g, (few, k), "bf16"), rand(g, (n, k), "bf16", k ** -0.5), rand(g, (n,), "bf16"), rand(g, (few, n), "bf16")
    want = x @ w.T   # in f32: both sides' sums are within the spread of the exact ones
    tol = 2 * (k + 20) * 2.0 ** -24 * (np.abs(x) @ np.abs(w).T + 1)
    again = lambda a: np.tile(a, (m // few, 1))  # noqa: E731
    xd, wd = up(again(x), "bf16"), up(w, "bf16")
    got = down(R.linear(xd, wd))
    assert np.all(np.abs(got[:few] - want) <= 2.0 ** -8 * np.abs(want) + tol)
    z = want + b
    full = z / (1 + np.exp(-z)) + r   # silu's slope stays below 1.1, its own error below 2^-18 of it
    fused = down(R.linear(xd, wd, up(b, "bf16"), "silu", up(again(r), "bf16")))
    assert np.all(np.abs(fused[:few] - full) <= 2.0 ** -8 * np.abs(full) + 2 * tol + 2.0 ** -18 * np.abs(z) + 2.0 ** -20)
    # every row block, against the first (a shared tile's sums are grouped in another way: 2 tol, one rounding)
    assert np.all(np.abs(got - again(got[:few])) <= 2.0 ** -7 * np.abs(again(want)) + 2 * again(tol))


def test_plan_is_what_runs(R, monkeypatch):
    """A product whose sums differ by tile and parts: the rule's name and parts, forced, give the bits of the call that is not."""
    m, k, n = 409, 5760, 8416
    g = np.random.Generator(np.random.PCG64(3))
    x, w = up(rand(g, (m, k), "bf16"), "bf16"), up(rand(g, (n, k), "bf16"), "bf16")
    tile, parts = plan(m, k, n)
    free = down(R.linear(x, w))
    monkeypatch.setenv("RAI_HIP_GEMM_TILE", tile)
    np.testing.assert_array_equal(free, down(R.linear_packed(x, w, k_splits=parts)))
    assert not np.array_equal(free, down(R.linear_packed(x, w, k_splits=parts + 1)))

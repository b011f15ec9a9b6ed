"""bf16 Linears of 2 to 32 rows where their streaming kernel changes form: four to ten K steps of 32 to a wave with the last ones beyond K, K in
two to nine parts, one, two and four tiles to a block, the last one past N; a fused norm and gated pairs, biases, two outputs, an f32 stream.  Weights in
fragment order, and with a norm, through the decoders that call them: one layer, held to the oracle by the bound that every bf16 decoder test
has.  Weights in rows also by themselves."""
import numpy as np
import pytest

from oracle import bezadra, phi2, qwen2
from tests import bezadra_models as bm
from tests.test_gpu_bezadra import deep_close
from tests.test_gpu_phi2 import make as make_phi2
from tests.test_gpu_qwen2_gemma import make
from tests.util import assert_close, down, rand, up

pytestmark = pytest.mark.gpu


def step(dec, ref, vocab, batch, what):
    ids = np.random.Generator(np.random.PCG64(batch)).integers(0, vocab, (batch, 2)).astype(np.uint32)
    for at in range(2):   # both calls are single tokens
        assert_close(dec.forward(ids[:, at:at + 1])[0], ref.fwd(ids[:, at:at + 1]), "bf16", what)
    dec.close()


@pytest.mark.parametrize("arch,width,ff,vocab,batch", [
    ("qwen2", 800, 2592, 1004, 9), ("qwen2", 1056, 4128, 5000, 16), ("gemma", 1312, 7168, 1004, 17), ("gemma", 1568, 2080, 8200, 31), ("qwen2", 2016, 2560, 4116, 32),
    ("qwen2", 2080, 16416, 500, 24), ("qwen2", 800, 2592, 1004, 2), ("gemma", 1056, 4128, 5000, 3), ("qwen2", 1568, 2080, 8200, 5), ("gemma", 2016, 7168, 1004, 8)])
def test_sequential_block(hip, arch, width, ff, vocab, batch):
    cfg = qwen2.Config(arch, vocab, width, ff, 1, 2, 1, "silu" if arch == "qwen2" else "gelu", max_position_embeddings=64, head_dim=64)
    dec, ref = make(cfg, "bf16", max_batch=batch, max_context=8)
    step(dec, ref, vocab, batch, f"{arch} {width} {ff} batch {batch}")


@pytest.mark.parametrize("heads,ff,batch", [(12, 2176, 11), (28, 5120, 27), (12, 5120, 2), (28, 2176, 7)])   # widths 960 and 2240, [dense | fc2] of 3136 and 7360
def test_parallel_block(hip, heads, ff, batch):
    cfg = phi2.Config(vocab_size=1000, hidden_size=heads * 80, intermediate_size=ff, num_hidden_layers=1, num_attention_heads=heads, max_position_embeddings=64)
    dec, ref = make_phi2(cfg, "bf16", hip, max_batch=batch, max_context=8)
    step(dec, ref, 1000, batch, f"phi2 {heads} heads batch {batch}")


@pytest.mark.parametrize("width,ff,batch", [(1024, 1888, 10), (1280, 2944, 32)])   # [o | down] of 1984 + 64 and 3072 columns onto the f32 stream
def test_f32_stream(hip, width, ff, batch):
    cfg = bm.config([bm.attention(heads=2, kv_heads=1, dim=64, vdim=64, ff=ff)], width=width, vocab=600, loop=(0, 1, 2))
    p = bezadra.random_params(cfg, "bf16", width)
    dec = bm.build(cfg, p, "bf16", max_batch=batch, max_context=8)
    ids = np.random.Generator(np.random.PCG64(ff)).integers(0, 600, (batch, 2)).astype(np.uint32)
    want = np.stack([bezadra.Model(cfg, p).logits(r) for r in ids])
    for at in range(2):
        deep_close(dec.forward(ids[:, at:at + 1])[0], want[:, at], "bf16", f"width {width}, step {at}")
    dec.close()


@pytest.fixture(scope="module")
def R(hip):
    from rai_amd import ops

    return ops


def spread(x, w):
    """K + 8 roundings of the absolute sum: any order of K f32 additions and the bias."""
    return (x.shape[1] + 8) * 2.0 ** -24 * (np.abs(x.astype(np.float64)) @ np.abs(w.astype(np.float64)).T + 1)


@pytest.mark.parametrize("m", [5, 8, 9, 16, 17, 32])
@pytest.mark.parametrize("k,n", [(800, 2052), (1056, 1500), (1568, 4100), (2080, 740), (2592, 3240), (4128, 2052), (7168, 1204), (8960, 4164), (2048, 8200)])
def test_rows_as_they_lie(R, m, k, n):
    g = np.random.Generator(np.random.PCG64(m * 1000 + k))
    x, w, r = rand(g, (m, k + 8), "bf16"), rand(g, (n, k + 16), "bf16", k ** -0.5), rand(g, (m, n), "bf16")
    x[:, k:], w[:, k:] = np.inf, np.nan   # behind the K of the views
    b = rand(g, (n,), "bf16")
    xd, wd = up(x, "bf16").narrow(1, 0, k), up(w, "bf16").narrow(1, 0, k)
    x, w = x[:, :k], w[:, :k]
    z = x.astype(np.float64) @ w.astype(np.float64).T + b
    full = z / (1 + np.exp(-z)) + r   # silu's slope stays below 1.1
    got = down(R.linear(xd, wd, up(b, "bf16"), "silu", up(r, "bf16"))).astype(np.float64)
    assert np.all(np.abs(got - full) <= 2.0 ** -8 * np.abs(full) + 2 * spread(x, w) + 2.0 ** -20)


@pytest.mark.parametrize("m,k,n,n1", [(6, 1600, 2056, 1028), (31, 2400, 1032, 4), (20, 3200, 1040, 516)])
def test_two_outputs(R, m, k, n, n1):
    g = np.random.Generator(np.random.PCG64(m + k))
    x, w = rand(g, (m, k), "bf16"), rand(g, (n, k), "bf16", k ** -0.5)
    b, b2 = rand(g, (n,), "bf16"), rand(g, (n,), "bf16")
    z = x.astype(np.float64) @ w.astype(np.float64).T + (b.astype(np.float64) + b2)
    want = np.concatenate([z[:, :n1], z[:, n1:] / (1 + np.exp(-z[:, n1:]))], 1)
    o1, o2 = R.linear_packed(up(x, "bf16"), up(w, "bf16"), bias=up(b, "bf16"), bias2=up(b2, "bf16"), act="silu", act_from=n1, n1=n1)
    got = np.concatenate([down(o1), down(o2)], 1).astype(np.float64)
    extra = 2.0 ** -23 * (np.abs(b) + np.abs(b2))
    assert np.all(np.abs(got - want) <= 2.0 ** -8 * np.abs(want) + 2 * spread(x, w) + extra + 2.0 ** -20)


@pytest.mark.parametrize("m,k,n", [(5, 1056, 1512), (16, 2048, 4112), (29, 1376, 8200)])
def test_gated(R, m, k, n):
    """gate, act(gate) and up each rounded: see test_few_rows_gated."""
    g = np.random.Generator(np.random.PCG64(m + n))
    x, w = rand(g, (m, k), "bf16"), rand(g, (n, k), "bf16", k ** -0.5)
    z = x.astype(np.float64) @ w.astype(np.float64).T
    gate, upv = z[:, 0::2], z[:, 1::2]
    want = gate / (1 + np.exp(-gate)) * upv
    got = down(R.linear_packed(up(x, "bf16"), up(w, "bf16"), act="silu", glu=True)).astype(np.float64)
    assert np.all(np.abs(got - want) <= 4 * 2.0 ** -8 * (np.abs(gate) + 1) * (np.abs(upv) + 1))


@pytest.mark.parametrize("m,k,n,taken", [(8, 1024, 1028, True), (9, 1024, 1028, False), (32, 2048, 2052, False), (16, 1024, 1032, True), (16, 736, 1028, False)])
def test_gated_columns_that_are_refused(R, m, k, n, taken):
    """Beyond eight rows gated products come in whole eights of columns, whichever kernel would serve them."""
    from rai_amd._lib import RaiHipError

    g = np.random.Generator(np.random.PCG64(m))
    x, w = up(rand(g, (m, k), "bf16"), "bf16"), up(rand(g, (n, k), "bf16"), "bf16")
    if taken:
        assert R.linear_packed(x, w, act="silu", glu=True).shape == (m, n // 2)
    else:
        with pytest.raises(RaiHipError, match="gated"):
            R.linear_packed(x, w, act="silu", glu=True)

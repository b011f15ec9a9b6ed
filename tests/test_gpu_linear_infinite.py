"""Infinite weights and activations where K is no whole number of what a block's waves take: what lies beyond K is made up from K's first columns, and must not
turn an infinite output into no number."""
import numpy as np
import pytest

from oracle import qwen2
from oracle.dtypes import rnd, to_storage
from tests.util import down, rand, up

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("m", [5, 8, 16, 32])
@pytest.mark.parametrize("k", [800, 896, 1056, 2336, 2592, 4128, 8960])
def test_rows_as_they_lie(hip, m, k):
    from rai_amd import ops

    g = np.random.Generator(np.random.PCG64(m * 1000 + k))
    n = 1536
    x, w = rand(g, (m, k), "bf16"), rand(g, (n, k), "bf16", k ** -0.5)
    x[x == 0], w[w == 0] = 1, 1
    w[3, 0], w[8, 31], w[n - 1, 0], w[700, 31] = np.inf, -np.inf, -np.inf, np.inf
    x[m - 1, 5] = np.inf
    with np.errstate(invalid="ignore"):
        want = x.astype(np.float64) @ w.astype(np.float64).T
    finite = np.isfinite(want)
    assert not np.isfinite(want[:, [3, 8, 700, n - 1]]).any() and finite.sum() == (m - 1) * (n - 4)
    for got in (ops.linear(up(x, "bf16"), up(w, "bf16")), ops.matmul(up(x, "bf16"), up(w, "bf16").transpose(0, 1))):
        got = down(got).astype(np.float64)
        assert np.array_equal(got[~finite], want[~finite], equal_nan=True)
        spread = (k + 8) * 2.0 ** -24 * (np.abs(x[:-1].astype(np.float64)) @ np.abs(np.where(np.isfinite(w), w, 0).astype(np.float64)).T)
        got, ref = np.where(finite, got, 0)[:-1], np.where(finite, want, 0)[:-1]
        assert np.all(np.abs(got - ref) <= 2.0 ** -8 * np.abs(ref) + 2 * spread)


@pytest.mark.parametrize("batch", [9, 16, 24])
@pytest.mark.parametrize("width,ff", [(800, 2592), (896, 4128), (1056, 2336)])
def test_fragments(hip, width, ff, batch):
    """The down projection of a layer (K whole or in parts) and the normed head of a batched step."""
    from rai_amd.models import Decoder

    vocab = 1004
    cfg = qwen2.Config("qwen2", vocab, width, ff, 1, 1, 1, "silu", max_position_embeddings=64, head_dim=64)
    params = qwen2.random_params(cfg, "bf16", seed=width)
    ids = np.arange(batch, dtype=np.uint32)[:, None]

    def run(params):
        dec = Decoder("qwen2", "bf16", vocab_size=vocab, hidden_size=width, intermediate_size=ff, num_hidden_layers=1, num_attention_heads=1,
                      num_key_value_heads=1, head_dim=64, rotary_dim=64, max_position_embeddings=64, hidden_act="silu", tie_word_embeddings=False, norm_eps=1e-6,
                      max_batch=batch, max_context=8)
        for name in dec.param_names():
            dec.load_param(name, to_storage(params[name], "bf16"))
        hidden, logits, _ = dec.forward_hidden(ids, want_logits=True)
        dec.close()
        return hidden[:, 0], logits

    hidden, logits = run(params)
    head = params["lm_head.weight"].copy()
    head[5, 0], head[17, 31], head[vocab - 1, 0] = np.inf, -np.inf, -np.inf
    got = run(params | {"lm_head.weight": head})[1]
    assert np.array_equal(np.isfinite(got), np.broadcast_to(~np.isin(np.arange(vocab), [5, 17, vocab - 1]), got.shape)) and not np.isnan(got).any()
    assert np.array_equal(np.sign(got[:, [5, 17, vocab - 1]]), np.sign(hidden[:, [0, 31, 0]]) * [1, -1, -1])   # the head's norm has positive weights
    assert np.array_equal(got[:, :5], logits[:, :5])
    w = params["model.layers.0.mlp.down_proj.weight"].copy()
    w[3, 0], w[width - 2, 31] = np.inf, -np.inf
    got = run(params | {"model.layers.0.mlp.down_proj.weight": rnd(w, "bf16")})[0]
    assert np.isinf(got[:, [3, width - 2]]).all()
    rest = ~np.isin(np.arange(width), [3, width - 2])
    assert np.array_equal(got[:, rest], hidden[:, rest])

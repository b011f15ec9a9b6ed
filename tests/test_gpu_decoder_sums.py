"""A decoder's results rest on the order of its f32 sums and on where it rounds: batched steps keep to both.  The logits of every family at batches on
either side of each kernel's range are held to their bits in tests/golden/decoder_sums.npz (written by make_decoder_sums.py there, which says
when), and the norm in front of a streamed Linear to one rounding of its result."""
from pathlib import Path

import numpy as np
import pytest

from oracle import bezadra, phi2, qwen2
from oracle.dtypes import rnd, to_storage
from tests import bezadra_models as bm
from tests.test_gpu_phi2 import make as make_phi2
from tests.test_gpu_qwen2_gemma import make

pytestmark = pytest.mark.gpu

GOLDEN = Path(__file__).parent / "golden" / "decoder_sums.npz"
VOCAB = 128


def seq(arch, width, ff, heads, kv_heads, dim):
    cfg = qwen2.Config(arch, VOCAB, width, ff, 1, heads, kv_heads, "silu" if arch == "qwen2" else "gelu", max_position_embeddings=64, head_dim=dim)
    return lambda batch: make(cfg, "bf16", max_batch=batch, max_context=8)[0]


def parallel(heads, ff):
    cfg = phi2.Config(vocab_size=VOCAB, hidden_size=heads * 80, intermediate_size=ff, num_hidden_layers=1, num_attention_heads=heads, max_position_embeddings=64)
    return lambda batch: make_phi2(cfg, "bf16", None, max_batch=batch, max_context=8)[0]


def hybrid(width, ff):
    cfg = bm.config([bm.attention(heads=2, kv_heads=1, dim=64, vdim=64, ff=ff)], width=width, vocab=VOCAB, loop=(0, 1, 2))
    return lambda batch: bm.build(cfg, bezadra.random_params(cfg, "bf16", width), "bf16", max_batch=batch, max_context=8)


# K of four to ten runs of eight steps and of two and three parts, whole and with a last run or a last part that is not
FAMILIES = {"gemma_2048": seq("gemma", 2048, 4096, 4, 1, 256), "qwen2_1536": seq("qwen2", 1536, 4480, 12, 2, 128), "qwen2_1568": seq("qwen2", 1568, 2592, 4, 2, 256),
            "phi2_2560": parallel(32, 2560), "phi2_960": parallel(12, 2176), "bezadra_1024": hybrid(1024, 1888)}
BATCHES = [2, 5, 8, 9, 16, 17, 32]


def logits(family, batch):
    """bf16 bits of the logits behind each of two tokens."""
    dec = FAMILIES[family](batch)
    ids = np.random.Generator(np.random.PCG64(batch)).integers(0, VOCAB, (batch, 2)).astype(np.uint32)
    got = np.stack([dec.forward(ids[:, at:at + 1])[0] for at in range(2)])
    dec.close()
    return to_storage(np.asarray(got, np.float32), "bf16")


@pytest.mark.parametrize("batch", BATCHES)
@pytest.mark.parametrize("family", FAMILIES)
def test_bits(hip, family, batch):
    got, want = logits(family, batch), np.load(GOLDEN)[f"{family}_{batch}"]
    assert got.shape == want.shape and np.array_equal(got, want), f"{(got != want).sum()} of {want.size} logits have other bits"


@pytest.mark.parametrize("batch", [2, 8, 9, 16, 17, 32])
@pytest.mark.parametrize("arch,width", [("qwen2", 1056), ("gemma", 1056), ("qwen2", 2048), ("gemma", 2048)])
def test_norm_rounds_once(hip, arch, width, batch):
    """No layer adds anything and the head reads single features, so that a logit is a feature of the normed embedding: x * scale * w (Gemma: 1 + w), rounded once
    from f32 whose `scale` may be off by the additions of its sum."""
    from rai_amd.models import Decoder

    g = np.random.Generator(np.random.PCG64(width + batch))
    vocab = batch + width
    table = np.concatenate([rnd(g.standard_normal((batch, width), dtype=np.float32), "bf16"), np.eye(width, dtype=np.float32)])
    dec = Decoder(arch, "bf16", vocab_size=vocab, hidden_size=width, intermediate_size=64, num_hidden_layers=1, num_attention_heads=1, num_key_value_heads=1,
                  head_dim=64, rotary_dim=64, max_position_embeddings=64, hidden_act="silu" if arch == "qwen2" else "gelu", tie_word_embeddings=True,
                  norm_eps=1e-6, max_batch=batch, max_context=8)
    w = rnd((arch == "qwen2") + 0.2 * g.standard_normal(width).astype(np.float32), "bf16")
    for name, size in dec.param_names().items():
        a = table if "embed" in name else w if name == "model.norm.weight" else np.zeros(size, np.float32)
        dec.load_param(name, to_storage(np.asarray(a, np.float32), "bf16"))
    got = np.asarray(dec.forward(np.arange(batch, dtype=np.uint32)[:, None])[0], np.float32)[:, batch:]
    dec.close()
    x = table[:batch]
    if arch == "gemma":
        x = rnd(x * rnd(np.float32(np.sqrt(width)), "bf16"), "bf16")
    scale = 1 / np.sqrt((x.astype(np.float64) ** 2).mean(1, keepdims=True) + 1e-6)
    wf = np.float32(1) + w if arch == "gemma" else w
    off = (width + 8) * 2.0 ** -24   # any order of the sum's additions, halved by the root, and the f32 steps behind it
    ends = [rnd((x * (scale * f).astype(np.float32) * wf).astype(np.float32), "bf16") for f in (1 - off, 1 + off)]
    assert np.all((got >= np.minimum(*ends)) & (got <= np.maximum(*ends)))

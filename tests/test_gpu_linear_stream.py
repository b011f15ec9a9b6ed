"""bf16 Linears of 9 to 32 rows on weights in fragment order, where their kernels change form, through the decoders that call them: four to ten K
steps of 32 to a wave with the last wave's beyond K, K in two to nine parts, one, two and four tiles to a block, the last one past N; a fused norm and
gated pairs, biases, two outputs, an f32 stream.  One layer, held to the oracle by the bound that every bf16 decoder test has."""
import numpy as np
import pytest

from oracle import bezadra, phi2, qwen2
from tests import bezadra_models as bm
from tests.test_gpu_bezadra import deep_close
from tests.test_gpu_phi2 import make as make_phi2
from tests.test_gpu_qwen2_gemma import make
from tests.util import assert_close

pytestmark = pytest.mark.gpu


def step(dec, ref, vocab, batch, what):
    ids = np.random.Generator(np.random.PCG64(batch)).integers(0, vocab, (batch, 2)).astype(np.uint32)
    for at in range(2):   # both calls are single tokens
        assert_close(dec.forward(ids[:, at:at + 1])[0], ref.fwd(ids[:, at:at + 1]), "bf16", what)
    dec.close()


@pytest.mark.parametrize("arch,width,ff,vocab,batch", [
    ("qwen2", 800, 2592, 1004, 9), ("qwen2", 1056, 4128, 5000, 16), ("gemma", 1312, 7168, 1004, 17), ("gemma", 1568, 2080, 8200, 31), ("qwen2", 2016, 2560, 4116, 32),
    ("qwen2", 2080, 16416, 500, 24)])
def test_sequential_block(hip, arch, width, ff, vocab, batch):
    cfg = qwen2.Config(arch, vocab, width, ff, 1, 2, 1, "silu" if arch == "qwen2" else "gelu", max_position_embeddings=64, head_dim=64)
    dec, ref = make(cfg, "bf16", max_batch=batch, max_context=8)
    step(dec, ref, vocab, batch, f"{arch} {width} {ff} batch {batch}")


@pytest.mark.parametrize("heads,ff,batch", [(12, 2176, 11), (28, 5120, 27)])   # widths 960 and 2240, [dense | fc2] of 3136 and 7360
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

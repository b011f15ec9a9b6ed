"""Grouped-query decode attention on both sides of the number of blocks up to which a block has eight waves: 256 of 128 features, 512 of 256 (256
where a block has 128 keys)."""
import numpy as np
import pytest

from oracle import qwen2
from tests.test_gpu_qwen2_gemma import make
from tests.util import assert_close

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dim,batch,keys", [(128, 42, "64"), (128, 43, "64"), (128, 43, "96"), (128, 43, "128"), (256, 42, "64"), (256, 43, "64"),
                                            (256, 86, "64"), (256, 43, "128"), (256, 65, "96")])
def test_decode_attention_of_many_sequences(hip, dim, batch, keys, monkeypatch):
    monkeypatch.setenv("RAI_HIP_ATTN_KEYS", keys)
    monkeypatch.setenv("RAI_HIP_ATTN_SPLITS", "2")   # or as many as the context takes
    cfg = qwen2.Config("qwen2", 200, 64, 96, 1, 12, 3, "silu", max_position_embeddings=160, head_dim=dim)
    dec, ref = make(cfg, "bf16", max_batch=batch, max_context=100 if keys == "64" else 150)
    ids = np.random.Generator(np.random.PCG64(dim + batch)).integers(0, cfg.vocab_size, (batch, 81)).astype(np.uint32)
    for step in range(3):
        logits, _ = dec.forward(ids)
        want = ref.fwd(ids)
        assert_close(logits, want, "bf16", f"step {step}")
        ids = np.argmax(want, -1).astype(np.uint32).reshape(batch, 1)
    dec.close()

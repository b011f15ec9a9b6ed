"""The single-row bf16 step where its launches change shape: widths that end inside a wave's 512 columns and every number of those
pieces up to eight; fewer pairs of rows than waves and many a wave; [o | down] rows of 1 to 21 pieces (20 are in flight); the delta
step with the MLP's first half beside it, and states too large for that."""
import numpy as np
import pytest

from oracle import bezadra
from tests import bezadra_models as bm
from tests.test_gpu_bezadra import deep_close, tokens

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("width,ff,heads,dim,vdim", [
    (64, 40, 1, 32, 32), (120, 200, 3, 20, 36), (512, 1000, 4, 64, 64), (576, 3000, 2, 32, 128), (1024, 520, 4, 128, 128), (1088, 4096, 4, 64, 64),
    (2048, 9000, 8, 128, 128), (2112, 9984, 4, 128, 128), (2600, 1024, 4, 64, 64), (4088, 512, 2, 64, 64), (256, 300, 2, 256, 256)])
def test_widths(hip, width, ff, heads, dim, vdim):
    cfg = bm.config([bm.delta(heads=heads, kv_heads=heads, dim=dim, vdim=vdim, conv=4, ff=ff), bm.attention(heads=4, kv_heads=2, ff=ff)], width=width, loop=(0, 1, 2))
    p = bezadra.random_params(cfg, "bf16", width)
    dec, ids = bm.build(cfg, p, "bf16", max_context=16), tokens(cfg, (1, 6), ff)
    want = np.stack([bezadra.Model(cfg, p).logits(r) for r in ids])
    got = bm.run_portions(dec, ids, [3, 1, 1, 1])
    deep_close(got, want[:len(got)], "bf16", f"width {width}, MLP {ff}")
    dec.close()

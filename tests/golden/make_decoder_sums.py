#!/usr/bin/env python3
"""Writes decoder_sums.npz beside this file: the bf16 logits of the decoders in tests/test_gpu_decoder_sums.py as the library now computes them.  The file
holds those of commit 039009d.  It is to be written again only where a change of the decoders' sums or roundings is meant.

    python tests/golden/make_decoder_sums.py [out.npz]     (needs a GPU)
"""
import sys
from pathlib import Path

import numpy as np

sys.path.insert(0, str(Path(__file__).resolve().parents[2]))

from rai_amd import _lib  # noqa: E402
from tests.test_gpu_decoder_sums import BATCHES, FAMILIES, GOLDEN, logits  # noqa: E402

_lib.call("rai_hip_init", 0)
np.savez_compressed(sys.argv[1] if len(sys.argv) > 1 else GOLDEN, **{f"{f}_{b}": logits(f, b) for f in FAMILIES for b in BATCHES})

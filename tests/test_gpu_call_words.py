"""The words a call exchanges with the device: token ids on either side of the count up to which kernels carry them."""
import numpy as np
import pytest

from rosylnalive_amd.gpu_core import HipBackend
from rosylnalive_amd.qwen import QwenConfig, QwenModel, synthetic_ids, synthetic_weights

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("t", [1, 255, 257, 1280, 1281, 1500])
def test_ids_reach_the_device(t):
    """A chunk of t ids gives the rows that chunks of 100 give (the float32 mode keeps a row's bits over any chunking)."""
    cfg = QwenConfig(1, 64, 4, 2, 16, 192, 512, 1500)
    w, ids = synthetic_weights(cfg, seed=3), synthetic_ids(3, "words", 1500, 512)[:t]
    rows, got = min(t, 100), []
    for chunk in (t, 100):
        b = HipBackend(0)
        m = QwenModel(b, cfg, mode="fp32", max_tokens=chunk)
        m.load_weights(w)
        logits, _ = m.forward(ids, 0, logits_rows=rows)
        got.append((logits.tobytes(), m.read_cache(0, "v", 0, t).tobytes()))
        m.close()
        b.close()
    assert got[0] == got[1]

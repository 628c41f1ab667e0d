"""The words a call exchanges with the device (token ids on either side of the count up to which kernels carry them), and its
command lists released before they are waited for."""
import numpy as np
import pytest

from gpu_session import Session
from rosylnalive_amd.gpu_core import DType, HipBackend
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


def test_one_shot_lists_released_before_the_wait():
    """A submission keeps nothing of its one-shot list: lists released, and their memory used again, before the waits."""
    n = 1 << 20
    x = np.arange(n, dtype=np.float32)
    t = {"x0": (DType.F32, (n,), 0, x)}
    t.update({f"x{i}": (DType.F32, (n,), 0, None) for i in range(1, 9)})
    s = Session(t)
    try:
        fences = []
        for i in range(8):
            cl = s.backend.begin()
            timer = cl.begin_timer(f"part {i}")
            cl.dispatch("scale_f32", s.fields("scale_f32", x=f"x{i}", y=f"x{i + 1}", n=n, a=2.0))
            cl.end_timer(timer)
            fences.append(s.backend.submit(cl))
            cl.release()
        for i, f in enumerate(fences):
            c = s.backend.wait(f)
            assert c.dispatches == 1 and [r.name for r in c.timers] == [f"part {i}"]
        assert np.array_equal(s.read("x8"), x * 256)
    finally:
        s.close()

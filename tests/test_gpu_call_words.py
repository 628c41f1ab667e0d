"""The words a call exchanges with the device (token ids on either side of the count up to which kernels carry them, the
decoded ids over many runs), and its command lists released before they are waited for."""
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


def test_decode_ids_over_many_runs():
    """decode_ids is the same however the steps are cut into runs: past 4,096 ids in all, after a run too long for the host
    words, between runs, after a new start, and after greedy (whose first id is the prefill's)."""
    cfg = QwenConfig(1, 1024, 16, 8, 128, 1024, 512, 1024)
    b = HipBackend(0)
    m = QwenModel(b, cfg, mode="fast", max_tokens=64, batch=8)
    m.load_weights(synthetic_weights(cfg, seed=9))
    for s in range(8):
        m.forward(synthetic_ids(9, f"ids{s}", 5, 512), 0, logits_rows=0, seq=s)

    def run(parts, look=False):
        m.decode_set(np.arange(8, dtype=np.int32), np.full(8, 5, np.int32))
        seen = []
        for i, n in enumerate(parts):
            m.decode_run(n)
            if look:
                seen.append(m.decode_ids(sum(parts[:i + 1]) * 8))
        return m.decode_ids(sum(parts) * 8), seen
    try:
        one = run([560])[0]  # one run of 4,480 ids: read back from the device
        many, seen = run([1, 2, 500, 40, 17], look=True)
        assert np.array_equal(many, one) and all(np.array_equal(x, one[:x.size]) for x in seen)
        assert np.array_equal(run([520, 40])[0], one)
        assert np.array_equal(run([3])[0], one[:24]) and np.array_equal(m.decode_ids(8), one[:8])
    finally:
        m.close()
        b.close()


@pytest.mark.parametrize("decode", ["persistent", "kernels"])
def test_greedy_then_decode_ids(decode, monkeypatch):
    monkeypatch.setenv("LRM_HIP_DECODE", decode)
    cfg = QwenConfig(1, 1024, 16, 8, 128, 3072, 512, 256)
    b = HipBackend(0)
    m = QwenModel(b, cfg, mode="fast", max_tokens=64)
    m.load_weights(synthetic_weights(cfg, seed=4))
    ids = synthetic_ids(4, "greedy", 20, 512)
    try:
        out = m.greedy(ids, 9)
        assert np.array_equal(m.decode_ids(9)[1:], out[1:])
        m.decode_run(3)  # from greedy's state
        longer = m.greedy(ids, 12)
        assert np.array_equal(longer[:9], out)
        _, first = m.forward(ids, 0, logits_rows=1)
        m.decode_set(first, 20)
        m.decode_run(4)
        m.decode_run(7)
        assert first == out[0] and np.array_equal(m.decode_ids(11), longer[1:])
    finally:
        m.close()
        b.close()

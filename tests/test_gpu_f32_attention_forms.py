"""attention_gqa_causal's matrix-core forms beside the general kernel (the same tensors one float off their alignment), bit for
bit: a decode row on either side of the workspace's size, a decode row dispatched with overlap (no workspace), and scores that
are NaN or infinite."""
import numpy as np
import pytest

from gpu_session import Session
from rosylnalive_amd.gpu_core import DType, TensorFlags
from test_gpu_f32_mfma import _attention

pytestmark = pytest.mark.gpu


def _same(a, b):
    nan = np.isnan(b)
    return np.array_equal(np.isnan(a), nan) and np.array_equal(np.where(nan, 0, a).view(np.uint32), np.where(nan, 0, b).view(np.uint32))


def _qkv(seed, rows, past, qh, kvh, hd):
    r = np.random.default_rng(seed)
    return [r.standard_normal((n, h * hd)).astype(np.float32) for n, h in ((rows, qh), (past + rows, kvh), (past + rows, kvh))]


# bytes of the row form: heads x blocks x (67 + dimensions) x 4, blocks = past / 64 + 1, of 4 MiB. 16 heads of 128: 336 blocks
# (past 21,503) fit, 337 do not; 32 heads of 64: 250 fit; 4 heads of 128: 1344 fit
@pytest.mark.parametrize("past,qh,kvh,hd", [(21503, 16, 8, 128), (21504, 16, 8, 128), (15999, 32, 8, 64), (16000, 32, 8, 64),
                                            (86015, 4, 4, 128), (86016, 4, 4, 128)])
def test_decode_row_at_the_workspace_size(past, qh, kvh, hd):
    blocks = past // 64 + 1
    assert (qh * blocks * (67 + hd) * 4 <= 4 << 20) == (past % 64 == 63)
    q, k, v = _qkv(past, 1, past, qh, kvh, hd)
    assert _same(_attention(q, k, v, qh, kvh, hd, past, 0), _attention(q, k, v, qh, kvh, hd, past, 1))


@pytest.mark.parametrize("past,qh,kvh,hd", [(700, 16, 8, 128), (40, 4, 2, 64), (1000, 4, 1, 16), (13, 16, 8, 128)])
def test_decode_row_overlapped(past, qh, kvh, hd):
    """Two overlapped rows and one on the main stream, which alone may use the workspace: all the same bits."""
    q, k, v = _qkv(past, 1, past, qh, kvh, hd)
    t = {n: (DType.F32, a.shape, TensorFlags.READ_ONLY, a) for n, a in (("q", q), ("k", k), ("v", v))}
    t.update({y: (DType.F32, q.shape, 0, None) for y in ("y0", "y1", "y2")})
    s = Session(t)
    try:
        f = dict(q="q", k="k", v="v", rows=1, q_row0=0, past=past, q_heads=qh, kv_heads=kvh, head_dim=hd, scale=float(hd ** -0.5))
        cl = s.backend.begin()
        cl.dispatch_overlapped("attention_gqa_causal", s.fields("attention_gqa_causal", y="y0", **f))
        cl.dispatch("attention_gqa_causal", s.fields("attention_gqa_causal", y="y1", **f))
        cl.dispatch_overlapped("attention_gqa_causal", s.fields("attention_gqa_causal", y="y2", **f))
        cl.barrier()
        s.backend.wait(s.backend.submit(cl))
        cl.release()
        y = [s.read(n) for n in ("y0", "y1", "y2")]
        assert np.isfinite(y[1]).all()
        assert y[0].tobytes() == y[1].tobytes() == y[2].tobytes()
    finally:
        s.close()


@pytest.mark.parametrize("rows,past,qh,kvh,hd", [(1, 200, 16, 8, 128), (1, 700, 4, 2, 16), (40, 150, 4, 2, 64),
                                                 (70, 100, 16, 8, 128), (1030, 70, 64, 32, 16)])
@pytest.mark.parametrize("kind", ["nan key", "inf key", "-inf key", "nan block", "-inf block", "-inf all", "inf query"])
def test_scores_that_are_not_finite(rows, past, qh, kvh, hd, kind):
    q, k, v = _qkv(rows + past, rows, past, qh, kvh, hd)
    q.reshape(rows, qh, hd)[:, :, 0] = 1.0  # dimension 0 of a key is its score's addend: the sign of an infinity there stays
    keys = k.reshape(past + rows, kvh, hd)
    at = {"nan key": (past // 2, np.nan), "inf key": (past // 2, np.inf), "-inf key": (past + rows // 2, -np.inf),
          "nan block": (slice(64, 128), np.nan), "-inf block": (slice(0, 64), -np.inf), "-inf all": (slice(None), -np.inf)}
    if kind in at:
        where, value = at[kind]
        keys[where, 0, 0] = value
    else:
        q.reshape(rows, qh, hd)[rows // 2, 0, 1] = np.inf
    tiled, general = _attention(q, k, v, qh, kvh, hd, past, 0), _attention(q, k, v, qh, kvh, hd, past, 1)
    assert _same(tiled, general)
    assert np.isnan(general).any() == (kind != "-inf key")

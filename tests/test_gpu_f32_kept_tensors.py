"""What a float32 forward leaves in the executor's activation tensors (QwenModel.token): the same bits with its fused
dispatches as with the separate ones (taps on), for a prompt with some and with all of its rows asked for, a chunked prompt
and a decode step; and catalog ids 45 and 46 against the dispatches they stand for."""
import ctypes as C
import struct

import numpy as np
import pytest

from gpu_session import Session
from oracle import cpuref
from rosylnalive_amd import _native
from rosylnalive_amd.gpu_core import DType, HipBackend, TensorFlags
from rosylnalive_amd.qwen import QwenConfig, QwenModel, synthetic_ids, synthetic_weights

pytestmark = pytest.mark.gpu

F32, BF16 = DType.F32, DType.BF16
RO = TensorFlags.READ_ONLY
CFG = QwenConfig(2, 256, 4, 2, 64, 448, 600, 192)
WIDTHS = {"x": 256, "h": 256, "oo": 256, "r": 256, "h2": 256, "dd": 256, "f": 256, "q": 256, "qn": 256, "qr": 256, "o": 256,
          "k": 128, "v": 128, "kn": 128, "kr": 128, "g": 448, "u": 448, "d": 448}


def _read(m, name, n):
    table = C.create_string_buffer(1 << 20)
    _native.check(_native.lib().lrm_hip_download(m.backend.handle, 0, 0, table, 1 << 20))
    row = struct.unpack_from("<16I", table.raw, m.token(name) * 64)
    raw = C.create_string_buffer(n * 4)
    _native.check(_native.lib().lrm_hip_download(m.backend.handle, row[0], row[1], raw, n * 4))
    return np.frombuffer(raw.raw, np.float32)


# (position, rows, logits rows) calls in turn; the tensors are read after the last
@pytest.mark.parametrize("calls", [((0, 90, 90),), ((0, 90, 3),), ((0, 130, 5),), ((0, 70, 1), (70, 1, 1))])
def test_activation_tensors(calls):
    w, ids = synthetic_weights(CFG, seed=5), synthetic_ids(5, "kept", 192, 600)
    got = []
    for taps in (True, False):
        b = HipBackend(0)
        m = QwenModel(b, CFG, mode="fp32", max_tokens=100, taps=taps)
        m.load_weights(w)
        try:
            for pos, t, lr in calls:
                m.forward(ids[pos:pos + t], pos, logits_rows=lr)
            rows = (t - 1) % 100 + 1  # of the last chunk
            got.append({n: _read(m, n, rows * c) for n, c in WIDTHS.items()})
            last = _read(m, "f_last", min(lr if not taps else rows, 100) * 256)
            got[-1]["f_last"] = last[-lr * 256:]
        finally:
            m.close()
            b.close()
    for n in got[0]:
        assert got[0][n].tobytes() == got[1][n].tobytes(), n
    assert got[1]["f_last"].tobytes() == got[1]["f"][-lr * 256:].tobytes()


def _f(r, *s):
    return r.standard_normal(s).astype(np.float32)


@pytest.mark.parametrize("rows,qh,kvh,hd,pos0", [(1, 16, 8, 128, 40), (5, 4, 2, 16, 0), (3, 3, 1, 258, 7), (2, 1, 1, 2, 3),
                                                 (2, 2, 1, 1024, 1)])
def test_qk_norm_rope_append_all(rows, qh, kvh, hd, pos0):
    r = np.random.default_rng(rows + hd)
    P, KC, QC, eps = pos0 + rows + 2, kvh * hd, qh * hd, 1e-6
    a = {"q": _f(r, rows, QC), "k": _f(r, rows, KC), "v": _f(r, rows, KC), "cos": _f(r, P, hd // 2), "sin": _f(r, P, hd // 2)}
    t = {n: (F32, x.shape, RO, x) for n, x in a.items()}
    t.update({n: (BF16, (hd,), RO, cpuref.bf16_narrow(_f(r, hd))) for n in ("wq", "wk")})
    for i in "12":
        t.update({n + i: (F32, s, 0, None) for n, s in (("qn", (rows, QC)), ("qr", (rows, QC)), ("kn", (rows, KC)),
                                                        ("kr", (rows, KC)), ("kc", (P, KC)), ("vc", (P, KC)))})
    names = ("qn", "qr", "kn", "kr", "kc", "vc")
    s = Session(t)
    try:
        got = s.run("qk_norm_rope_append_all", [n + "1" for n in names], q="q", k="k", v="v", q_norm="wq", k_norm="wk",
                    cos_table="cos", sin_table="sin", qn="qn1", qr="qr1", kn="kn1", kr="kr1", k_cache="kc1", v_cache="vc1",
                    rows=rows, q_heads=qh, kv_heads=kvh, head_dim=hd, pos0=pos0, eps=eps)
        cp = dict(rows=rows, cols=KC, src_row0=0, dst_row0=pos0, src_stride=KC, dst_stride=KC)
        ref = s.run_list([
            ("rmsnorm_rows", dict(x="q", w="wq", y="qn2", rows=rows * qh, cols=hd, eps=eps)),
            ("rmsnorm_rows", dict(x="k", w="wk", y="kn2", rows=rows * kvh, cols=hd, eps=eps)),
            ("rope_apply", dict(x="qn2", cos_table="cos", sin_table="sin", y="qr2", rows=rows * qh, heads=qh, head_dim=hd, pos0=pos0)),
            ("rope_apply", dict(x="kn2", cos_table="cos", sin_table="sin", y="kr2", rows=rows * kvh, heads=kvh, head_dim=hd, pos0=pos0)),
            ("copy_rows", dict(src="kr2", dst="kc2", **cp)), ("copy_rows", dict(src="v", dst="vc2", **cp))],
            [n + "2" for n in names])
        for n in names:
            assert got[n + "1"].tobytes() == ref[n + "2"].tobytes(), n
    finally:
        s.close()


@pytest.mark.parametrize("rows,cols,tail", [(1, 1, 1), (7, 64, 3), (3, 255, 3), (2, 2048, 1), (5, 2049, 2), (2, 5000, 2)])
def test_add_rmsnorm_rows_tail(rows, cols, tail):
    r = np.random.default_rng(rows + cols)
    a, b, w = _f(r, rows, cols), _f(r, rows, cols), cpuref.bf16_narrow(_f(r, cols))
    t = {"a": (F32, a.shape, RO, a), "b": (F32, a.shape, RO, b), "w": (BF16, w.shape, RO, w), "last": (F32, (tail, cols), 0, None)}
    t.update({n: (F32, a.shape, 0, None) for n in ("r", "y", "r2", "y2")})
    s = Session(t)
    try:
        got = s.run("add_rmsnorm_rows_tail", ["r", "y", "last"], a="a", b="b", w="w", r="r", y="y", y_tail="last", rows=rows,
                    cols=cols, eps=1e-6, tail=tail)
        ref = s.run_list([("add", dict(a="a", b="b", y="r2", n=rows * cols)),
                          ("rmsnorm_rows", dict(x="r2", w="w", y="y2", rows=rows, cols=cols, eps=1e-6))], ["r2", "y2"])
        assert got["r"].tobytes() == ref["r2"].tobytes() and got["y"].tobytes() == ref["y2"].tobytes()
        assert got["last"].tobytes() == ref["y2"][-tail:].tobytes()
    finally:
        s.close()

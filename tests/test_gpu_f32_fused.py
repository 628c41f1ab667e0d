"""The float32 fusions (catalog ids 41..44) equal the reference dispatches they stand for bit for bit, at the sizes where a
tile, a register set or a block ends, and under the reference kernel set; the fp32 executor gives the same logits with its
taps on (the separate dispatches) and off (the fusions)."""
import numpy as np
import pytest

from gpu_session import Session
from oracle import cpuref
from rosylnalive_amd.gpu_core import DType, HipBackend, TensorFlags
from rosylnalive_amd.qwen import QwenConfig, QwenModel, synthetic_ids, synthetic_weights

pytestmark = pytest.mark.gpu

F32, BF16, U32 = DType.F32, DType.BF16, DType.U32
RO = TensorFlags.READ_ONLY


def _f(r, *s):
    return r.standard_normal(s).astype(np.float32)


@pytest.mark.parametrize("m,ns,k", [(1, (2048, 1024, 1024), 1024), (3, (1, 16, 17), 72), (17, (33, 64, 31), 129),
                                    (150, (2048, 1024, 1000), 256), (300, (4000, 3000), 64), (2, (48, 16400), 64),
                                    (40, (100, 7), 33)])
def test_matmul_groups(m, ns, k):
    r = np.random.default_rng(m + k)
    x, ws = _f(r, m, k), [cpuref.bf16_narrow(_f(r, n, k) * 0.1) for n in ns]
    t = {"x": (F32, x.shape, 0, x)}
    for i, w in enumerate(ws):
        t.update({f"w{i}": (BF16, w.shape, RO, w), f"y{i}": (F32, (m, ns[i]), 0, None), f"z{i}": (F32, (m, ns[i]), 0, None)})
    s = Session(t)
    try:
        f = {"x": "x", "m": m, "k": k}
        for i, n in enumerate(ns):
            f.update({f"w{i}": f"w{i}", f"y{i}": f"y{i}", f"n{i}": n})
        got = s.run("matmul_bf16w_triple" if len(ns) == 3 else "matmul_bf16w_pair", [f"y{i}" for i in range(len(ns))], **f)
        for i, n in enumerate(ns):
            one = s.run("matmul_bf16w", [f"z{i}"], x="x", w=f"w{i}", y=f"z{i}", m=m, n=n, k=k)[f"z{i}"]
            assert got[f"y{i}"].tobytes() == one.tobytes(), i
    finally:
        s.close()


@pytest.mark.parametrize("rows,qh,kvh,hd,pos0", [(1, 16, 8, 128, 40), (5, 4, 2, 16, 0), (3, 3, 1, 258, 7), (2, 1, 1, 2, 3)])
def test_qk_norm_rope_append(rows, qh, kvh, hd, pos0):
    r = np.random.default_rng(rows + hd)
    P, KC = pos0 + rows + 2, kvh * hd
    a = {"q": _f(r, rows, qh * hd), "k": _f(r, rows, KC), "v": _f(r, rows, KC), "cos": _f(r, P, hd // 2), "sin": _f(r, P, hd // 2)}
    t = {n: (F32, x.shape, RO, x) for n, x in a.items()}
    for n in ("qn", "kn"):
        t[n] = (BF16, (hd,), RO, cpuref.bf16_narrow(_f(r, hd)))
    for n, c in (("qr", (rows, qh * hd)), ("kc", (P, KC)), ("vc", (P, KC)), ("q1", (rows, qh * hd)), ("k1", (rows, KC)),
                 ("q2", (rows, qh * hd)), ("k2", (rows, KC)), ("kc2", (P, KC)), ("vc2", (P, KC))):
        t[n] = (F32, c, 0, None)
    s = Session(t)
    try:
        eps = 1e-6
        got = s.run("qk_norm_rope_append", ["qr", "kc", "vc"], q="q", k="k", v="v", q_norm="qn", k_norm="kn",
                    cos_table="cos", sin_table="sin", qr="qr", k_cache="kc", v_cache="vc", rows=rows, q_heads=qh,
                    kv_heads=kvh, head_dim=hd, pos0=pos0, eps=eps)
        ref = s.run_list([
            ("rmsnorm_rows", dict(x="q", w="qn", y="q1", rows=rows * qh, cols=hd, eps=eps)),
            ("rmsnorm_rows", dict(x="k", w="kn", y="k1", rows=rows * kvh, cols=hd, eps=eps)),
            ("rope_apply", dict(x="q1", cos_table="cos", sin_table="sin", y="q2", rows=rows * qh, heads=qh, head_dim=hd, pos0=pos0)),
            ("rope_apply", dict(x="k1", cos_table="cos", sin_table="sin", y="k2", rows=rows * kvh, heads=kvh, head_dim=hd, pos0=pos0)),
            ("copy_rows", dict(src="k2", dst="kc2", rows=rows, cols=KC, src_row0=0, dst_row0=pos0, src_stride=KC, dst_stride=KC)),
            ("copy_rows", dict(src="v", dst="vc2", rows=rows, cols=KC, src_row0=0, dst_row0=pos0, src_stride=KC, dst_stride=KC)),
        ], ["q2", "kc2", "vc2"])
        assert got["qr"].tobytes() == ref["q2"].tobytes()
        assert got["kc"].tobytes() == ref["kc2"].tobytes() and got["vc"].tobytes() == ref["vc2"].tobytes()
    finally:
        s.close()


@pytest.mark.parametrize("rows,cols", [(1, 1), (7, 64), (3, 255), (2, 2048), (2, 2049), (1, 5000)])
def test_add_rmsnorm_rows(rows, cols):
    r = np.random.default_rng(rows + cols)
    a, b, w = _f(r, rows, cols), _f(r, rows, cols), cpuref.bf16_narrow(_f(r, cols))
    t = {"a": (F32, a.shape, RO, a), "b": (F32, a.shape, RO, b), "w": (BF16, w.shape, RO, w)}
    t.update({n: (F32, a.shape, 0, None) for n in ("r", "y", "r2", "y2")})
    s = Session(t)
    try:
        got = s.run("add_rmsnorm_rows", ["r", "y"], a="a", b="b", w="w", r="r", y="y", rows=rows, cols=cols, eps=1e-6)
        ref = s.run_list([("add", dict(a="a", b="b", y="r2", n=rows * cols)),
                          ("rmsnorm_rows", dict(x="r2", w="w", y="y2", rows=rows, cols=cols, eps=1e-6))], ["r2", "y2"])
        assert got["r"].tobytes() == ref["r2"].tobytes() and got["y"].tobytes() == ref["y2"].tobytes()
    finally:
        s.close()


@pytest.mark.parametrize("cols", [1, 1000, 1024, 1025, 4096, 4097, 9000])
def test_argmax_rows_block_edges(cols):
    r = np.random.default_rng(cols)
    x = np.round(_f(r, 6, cols) * 4)  # ties
    x[1] = -np.inf
    x[2, cols // 2] = np.nan
    x[3, cols - 1] = 1e9
    s = Session({"x": (F32, x.shape, RO, x), "y": (U32, (6,), 0, None)})
    try:
        y = s.run("argmax_rows", ["y"], x="x", y="y", rows=6, cols=cols)["y"]
        ref = np.argmax(x, 1).astype(np.uint32)
        ref[2] = 0xFFFFFFFF
        assert y.tolist() == ref.tolist()
    finally:
        s.close()


def test_fp32_forward_equals_its_separate_dispatches():
    cfg = QwenConfig(2, 256, 4, 2, 64, 448, 600, 192)
    w, ids = synthetic_weights(cfg, seed=5), synthetic_ids(5, "fused", 130, 600)
    out = []
    for taps in (True, False):
        b = HipBackend(0)
        b.load_kernels()  # the reference set
        assert b.contains(41) and b.contains(44)
        m = QwenModel(b, cfg, mode="fp32", max_tokens=100, taps=taps)
        m.load_weights(w)
        rows = [m.forward(ids[:100], 0, logits_rows=100)[0], m.forward(ids[100:129], 100, logits_rows=3)[0],
                m.forward(ids[129:], 129)[0], m.read_cache(1, "k", 0, 130), m.read_cache(1, "v", 0, 130)]
        out.append(b"".join(np.ascontiguousarray(x).tobytes() for x in rows))
        m.close()
        b.close()
    assert out[0] == out[1]


def test_decode_ids_come_back_across_runs_and_past_the_host_words():
    """decode_ids after one run, after more, past what the host keeps (4,096 words) and with the state's tensors exposed
    give the same ids."""
    cfg = QwenConfig(1, 1024, 16, 8, 128, 1024, 512, 1024)
    w = synthetic_weights(cfg, seed=9)
    b = HipBackend(0)
    m = QwenModel(b, cfg, mode="fast", max_tokens=64, batch=8)
    m.load_weights(w)
    for s in range(8):
        m.forward(synthetic_ids(9, f"ids{s}", 5, 512), 0, logits_rows=0, seq=s)
    try:
        def run(parts):
            m.decode_set(np.arange(8, dtype=np.int32), np.full(8, 5, np.int32))
            for n in parts:
                m.decode_run(n)
            return m.decode_ids(sum(parts) * 8)
        one = run([520])  # 4,160 ids: read back from the device
        two = run([3, 500])
        assert np.array_equal(one[:503 * 8], two)
        m.token("dec.state")
        assert np.array_equal(run([3, 500]), two)
    finally:
        m.close()
        b.close()

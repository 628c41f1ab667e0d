"""Which tile or loop a fast GEMM takes, and whether a decode GEMV's wave takes one row or two, changes no bit of a result: the
rows of a call equal the first rows of a larger one that takes other forms (the rules' tile counts are in the comments), bit
for bit."""
import numpy as np
import pytest

from gpu_session import Session
from oracle import cpuref
from rosylnalive_amd.gpu_core import DType, TensorFlags

pytestmark = pytest.mark.gpu

F32, F16, BF16 = DType.F32, DType.F16, DType.BF16
RO = TensorFlags.READ_ONLY


def _half(r, *s, scale=1.0):
    return (r.standard_normal(s) * scale).astype(np.float16).view(np.uint16)


# 64 rows and half columns; 64 rows; 128 rows; the direct-to-LDS loop (512 tiles)
@pytest.mark.parametrize("n,k,ms", [(65536, 64, (5, 64, 65, 128)), (4099, 192, (1, 64, 100, 129, 300, 512))])
def test_gemm_f32(n, k, ms):
    r = np.random.default_rng(n)
    a, w = _half(r, ms[-1], k), _half(r, n, k, scale=0.05)
    s = Session({"a": (F16, a.shape, 0, a), "w": (F16, w.shape, RO, w), "y": (F32, (ms[-1], n), 0, None)})
    try:
        y = [s.run("gemm_f32", ["y"], a="a", w="w", y="y", m=m, n=n, k=k)["y"][:m] for m in ms]
        for g in y:
            assert np.array_equal(g.view(np.uint32), y[-1][:len(g)].view(np.uint32)), len(g)
    finally:
        s.close()


# 3072: half columns (up to 128 rows), 64 rows (257 and 500), 96 pairs on the direct loop (1000: 256 tiles, 1500: 384), 64 pairs
# (2048: 768). 4864: counts that 8 does not divide (448: 304, 532 or 1064 tiles)
@pytest.mark.parametrize("inter,ms", [(3072, (1, 64, 128, 257, 500, 1000, 1500, 2048)), (4864, (37, 129, 448, 513, 700)),
                                      (200, (5, 65, 300))])
def test_gemm_swiglu(inter, ms):
    r = np.random.default_rng(inter)
    a, w = _half(r, ms[-1], 128), _half(r, 2 * inter, 128, scale=0.05)
    s = Session({"a": (F16, a.shape, 0, a), "w": (F16, w.shape, RO, w), "y": (F16, (ms[-1], inter), 0, None)})
    try:
        y = [s.run("gemm_swiglu", ["y"], a="a", w="w", y="y", m=m, inter=inter, k=128, a_shift=0)["y"][:m] for m in ms]
        for g in y:
            assert np.array_equal(g, y[-1][:len(g)]), len(g)
    finally:
        s.close()


# (17 rows and up: fewer take the skinny form) 64 x 32, 64 x 64, 128 x 64 and direct-to-LDS tiles; the last two of splits under
# 512 k, with two rounds of 64 rows
@pytest.mark.parametrize("n,k,splits,ms", [(1024, 1024, 2, (17, 64, 300, 500, 513, 777, 1500)), (1000, 1536, 1, (33, 600, 2000)),
                                           (2048, 2048, 4, (20, 129, 400, 700, 840)), (1000, 512, 2, (50, 576, 900)),
                                           (96, 128, 2, (17, 1000))])
def test_gemm_residual_split(n, k, splits, ms):
    r = np.random.default_rng(n + k)
    a, w = _half(r, ms[-1], k), _half(r, n, k, scale=0.05)
    s = Session({"a": (F16, a.shape, 0, a), "w": (F16, w.shape, RO, w), "p": (F32, (splits * ms[-1], n), 0, None)})
    try:
        p = []
        for m in ms:
            g = s.run("gemm_residual_split", ["p"], a="a", w="w", partials="p", m=m, n=n, k=k, splits=splits)["p"]
            p.append(g.ravel()[:splits * m * n].reshape(splits, m, n))
        for g in p:
            assert np.array_equal(g.view(np.uint32), p[-1][:, :g.shape[1]].view(np.uint32)), g.shape
    finally:
        s.close()


# 32 heads: 64 rows (up to 512), 128 rows (513 to 1408), the direct-to-LDS loop (1409: 384 tiles; 1900: 480); 12 heads: 64
# and 128 rows
@pytest.mark.parametrize("qh,ms", [(16, (1, 64, 300, 512, 513, 1300, 1409, 1900)), (6, (70, 1000, 2000))])
def test_gemm_qkv_rope(qh, ms):
    r = np.random.default_rng(qh)
    hid, kvh, mp, M = 128, qh // 2, 2048, ms[-1]
    a, w = _half(r, M, hid), _half(r, (qh + 2 * kvh) * 128, hid, scale=0.1)
    nw = [cpuref.bf16_narrow(1 + 0.1 * r.standard_normal(128)) for _ in range(2)]
    cs = [r.standard_normal((mp, 64)).astype(np.float32) for _ in range(2)]
    s = Session({"h": (F16, a.shape, 0, a), "w": (F16, w.shape, RO, w), "qn": (BF16, (128,), RO, nw[0]),
                 "kn": (BF16, (128,), RO, nw[1]), "c": (F32, (mp, 64), RO, cs[0]), "s": (F32, (mp, 64), RO, cs[1]),
                 "q": (F16, (M, qh * 128), 0, None), "kc": (F16, (kvh, mp, 128), 0, None), "vc": (F16, (kvh, mp // 64, 128, 64), 0, None)})
    try:
        out = []
        for m in ms:
            g = s.run("gemm_qkv_rope", ["q", "kc", "vc"], h="h", w="w", q_norm="qn", k_norm="kn", cos_table="c", sin_table="s",
                      q="q", k_cache="kc", v_cache="vc", m=m, hidden=hid, q_heads=qh, kv_heads=kvh, pos0=0, max_pos=mp, eps=1e-6)
            v = g["vc"].transpose(0, 1, 3, 2).reshape(kvh, mp, 128)
            out.append((g["q"][:m], g["kc"][:, :m], v[:, :m]))
        for (q, k, v), m in zip(out, ms):
            assert np.array_equal(q, out[-1][0][:m]) and np.array_equal(k, out[-1][1][:, :m]) and np.array_equal(v, out[-1][2][:, :m]), m
    finally:
        s.close()


@pytest.mark.parametrize("k", [1032, 1536, 2048])
def test_gemv_two_rows_per_wave(k):
    """4097 rows or pairs take two per wave, 900 one."""
    r = np.random.default_rng(k)
    n, few = 4097, 900
    x, nw = r.standard_normal(k).astype(np.float32), cpuref.bf16_narrow(1 + 0.1 * r.standard_normal(k))
    w = cpuref.bf16_narrow((r.standard_normal((2 * n, k)) * 0.05).astype(np.float32))
    wf = np.concatenate([w[:few], w[n:n + few]])
    s = Session({"x": (F32, (k,), RO, x), "nw": (BF16, (k,), RO, nw), "w": (BF16, w.shape, RO, w), "wf": (BF16, wf.shape, RO, wf),
                 "y": (F32, (n,), 0, None), "yf": (F32, (few,), 0, None)})
    try:
        for kernel, f in (("gemv_norm_dec", "n"), ("gemv_swiglu_dec", "inter")):
            c = dict(x="x", norm="nw", eps=1e-6, **{"k" if f == "n" else "hidden": k})
            two = s.run(kernel, ["y"], w="w", y="y", **{f: n}, **c)["y"]
            one = s.run(kernel, ["yf"], w="wf", y="yf", **{f: few}, **c)["yf"]
            assert np.array_equal(two[:few].view(np.uint32), one.view(np.uint32)), kernel
    finally:
        s.close()

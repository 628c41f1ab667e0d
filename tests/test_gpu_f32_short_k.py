"""matmul_bf16w and its grouped forms for short k: k = 0 writes +0 and reads nothing (x and w are one element here), every
other equals CpuRef F32 bit for bit; at the row and column counts of each tile form, and at the k where the form changes: the
short kernel's stages (16, 32, 64) and limits, tiles that end inside a group or with it, whole groups."""
import numpy as np
import pytest

from gpu_session import Session
from oracle import cpuref
from rosylnalive_amd.gpu_core import DType, TensorFlags

pytestmark = pytest.mark.gpu

F32, BF16 = DType.F32, DType.BF16
RO = TensorFlags.READ_ONLY


@pytest.mark.parametrize("m,ns", [(1, (1,)), (1, (17,)), (16, (16500,)), (17, (33,)), (700, (3000,)), (3, (40, 7)),
                                  (40, (100, 33)), (1, (16, 1, 65)), (150, (64, 31, 200))])
@pytest.mark.parametrize("k", [0, 1, 7, 8, 9, 16, 17, 32, 33, 40, 64, 65, 72, 128, 129, 200, 257, 384, 385, 392, 504, 511, 520])
def test_matmul_short_k(m, ns, k):
    r = np.random.default_rng(m + k)
    x = r.standard_normal((m, max(k, 1)))[:, :k].astype(np.float32) if k else np.zeros((m, 0), np.float32)
    ws = [cpuref.bf16_narrow(r.standard_normal((n, k)).astype(np.float32)) for n in ns]
    one = np.full(1, np.nan, np.float32)
    t = {"x": (F32, x.shape, RO, x) if k else (F32, (1,), RO, one)}
    for i, (n, w) in enumerate(zip(ns, ws)):
        t[f"w{i}"] = (BF16, w.shape, RO, w) if k else (BF16, (2,), RO, np.full(2, 0x7FC0, np.uint16))
        t[f"y{i}"] = (F32, (m, n), 0, None)
    s = Session(t)
    try:
        if len(ns) == 1:
            got = s.run("matmul_bf16w", ["y0"], x="x", w="w0", y="y0", m=m, n=ns[0], k=k)
        else:
            f = {"x": "x", "m": m, "k": k}
            for i, n in enumerate(ns):
                f.update({f"w{i}": f"w{i}", f"y{i}": f"y{i}", f"n{i}": n})
            got = s.run("matmul_bf16w_pair" if len(ns) == 2 else "matmul_bf16w_triple", [f"y{i}" for i in range(len(ns))], **f)
        for i, n in enumerate(ns):
            ref = cpuref.matmul_bf16w(x, ws[i]) if k else np.zeros((m, n), np.float32)
            assert got[f"y{i}"].tobytes() == ref.tobytes(), i
    finally:
        s.close()


@pytest.mark.parametrize("m,n,k", [(1, 65537, 64), (3, 65540, 80), (1, 65537, 88), (2, 65600, 319), (1, 65537, 321),
                                   (40, 20000, 32), (40, 20000, 40), (33, 20001, 33), (40, 20000, 127), (40, 20000, 130)])
def test_matmul_short_k_of_many_tiles(m, n, k):
    r = np.random.default_rng(m + k)
    x = r.standard_normal((m, k)).astype(np.float32)
    w = cpuref.bf16_narrow(r.standard_normal((n, k)).astype(np.float32))
    s = Session({"x": (F32, x.shape, RO, x), "w": (BF16, w.shape, RO, w), "y": (F32, (m, n), 0, None)})
    try:
        y = s.run("matmul_bf16w", ["y"], x="x", w="w", y="y", m=m, n=n, k=k)["y"]
        assert y.tobytes() == cpuref.matmul_bf16w(x, w).tobytes()
    finally:
        s.close()

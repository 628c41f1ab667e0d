"""The float32 contractions on the matrix cores (kernels_f32.hip) at the sizes where their tiles end.

- matmul_bf16w: every tile (16 x 16 and 16 x 32 up to 16 rows, 32 x 32 and 64 x 64 above; 16-byte and element loads) at
  remainders of rows, columns and k equals CpuRef F32 bit for bit, rows whose products underflow to -0 included (the
  padding past k must keep a chain's -0).
- attention_gqa_causal: the matrix-core kernel (16-byte aligned tensors, head_dim 16, 32, 64, 128) equals the general
  kernel, which the same tensors one float off their alignment take, bit for bit: one wave per tile and eight, tiles that
  end inside a row's heads, block edges, the single query row's three launches up to the end of their workspace, and an
  infinity or NaN among the values of keys past a query's own, which only the queries that own them may see.
"""
import numpy as np
import pytest

from gpu_session import Session
from oracle import cpuref
from rosylnalive_amd.gpu_core import Arena, ArgBlock, DType, HeapPlanner, HipBackend, TensorFlags, TensorTable

pytestmark = pytest.mark.gpu

F32, BF16 = DType.F32, DType.BF16
RO = TensorFlags.READ_ONLY


@pytest.mark.parametrize("m,n,k", [(1, 1, 8), (1, 31, 136), (2, 33, 520), (2, 65, 1000), (1, 40, 129), (3, 64, 64),
                                   (16, 65, 72), (17, 100, 200), (33, 31, 1000), (37, 96, 1028), (700, 3000, 72),
                                   (700, 3000, 67)])
def test_matmul_tiles_are_cpuref_f32(m, n, k):
    r = np.random.default_rng(m * 7 + n * 3 + k)
    x = r.standard_normal((m, k)).astype(np.float32)
    x[m // 2] *= np.float32(1e-38)  # products under 2^-149: sums of +0 and -0
    w = cpuref.bf16_narrow(r.standard_normal((n, k)) * 1e-8)
    s = Session({"x": (F32, x.shape, 0, x), "w": (BF16, w.shape, RO, w), "y": (F32, (m, n), 0, None)})
    try:
        y = s.run("matmul_bf16w", ["y"], x="x", w="w", y="y", m=m, n=n, k=k)["y"]
        assert y.tobytes() == cpuref.matmul_bf16w(x, w).tobytes()
    finally:
        s.close()


def _attention(q, k, v, qh, kvh, hd, past, shift):
    """attention_gqa_causal over tensors that start `shift` floats into their placements."""
    b = HipBackend(0)
    try:
        b.load_kernels()
        arrays = {"q": q, "k": k, "v": v, "y": np.full_like(q, np.float32(7))}
        planner, places = HeapPlanner(), {}
        for n, a in arrays.items():
            places[n] = planner.allocate(Arena.ACTIVATIONS, a.nbytes + 64)
        layout = planner.build()
        heap, table, tok = b.create_heap(layout), TensorTable(layout), {}
        for n, a in arrays.items():
            whole = table.add_placed(n + ".whole", places[n], F32, [a.size + 16], 0)
            tok[n] = table.add_view(n, whole, [a.size], shift)
        sealed = table.seal()
        heap.write_table(sealed)
        for n, a in arrays.items():
            r = sealed.row(tok[n])
            heap.upload(r[0], r[1], a)
        rows = q.shape[0]
        cl = b.begin()
        cl.dispatch("attention_gqa_causal", ArgBlock.encode(
            "attention_gqa_causal", q=tok["q"], k=tok["k"], v=tok["v"], y=tok["y"], rows=rows, q_row0=0, past=past,
            q_heads=qh, kv_heads=kvh, head_dim=hd, scale=float(np.float32(hd ** -0.5))))
        b.wait(b.submit(cl))
        cl.release()
        r = sealed.row(tok["y"])
        return np.frombuffer(heap.download(r[0], r[1], q.nbytes), np.float32).reshape(q.shape)
    finally:
        b.close()


@pytest.mark.parametrize("rows,past,qh,kvh,hd,odd", [
    (1, 0, 4, 2, 16, False), (1, 56, 4, 2, 16, False), (17, 47, 6, 2, 32, False), (5, 59, 8, 1, 64, False),
    (1, 63, 16, 8, 128, False), (1, 700, 16, 8, 128, False), (1, 64, 4, 4, 128, False), (1, 5000, 8, 2, 64, False),
    (1, 511, 4, 2, 16, False), (1, 448, 4, 1, 32, False), (1, 21500, 16, 8, 128, False), (150, 0, 16, 8, 128, False),
    (9, 1015, 16, 8, 128, False), (1030, 0, 16, 8, 128, False),
    (1030, 0, 64, 32, 16, False), (270, 3, 512, 128, 32, False), (70, 30, 4, 2, 64, True), (40, 500, 16, 8, 128, True),
    (1030, 5, 64, 32, 16, True)])
def test_attention_equals_the_general_kernel(rows, past, qh, kvh, hd, odd):
    r = np.random.default_rng(rows + past + hd)
    keys = past + rows
    q, k, v = (r.standard_normal((n, h * hd)).astype(np.float32) for n, h in ((rows, qh), (keys, kvh), (keys, kvh)))
    if odd:  # values that only the queries from that key on may see
        v[keys - 1, 0] = np.nan
        v[past + rows // 2, hd - 1] = np.inf
        v[past + rows // 3, 1] = -np.inf
    tiled, general = _attention(q, k, v, qh, kvh, hd, past, 0), _attention(q, k, v, qh, kvh, hd, past, 1)
    nan = np.isnan(general)
    assert np.array_equal(np.isnan(tiled), nan) and nan.any() == odd
    assert np.array_equal(np.where(nan, 0, tiled).view(np.uint32), np.where(nan, 0, general).view(np.uint32))
    if odd:
        assert np.isfinite(tiled[:rows // 3]).all()

"""The prefill GEMMs' smaller tiles (64 rows; 64 rows and half the columns) where the rule of rounds picks them: one to a few
row tiles, partial in rows and columns, against float64 on the same fp16 inputs. The sums are float32 (1e-6 relative in the
2-norm, as the other tiles' tests); gemm_swiglu rounds its products to fp16 (2^-11 of each value at most, 2.9e-4 in the
2-norm) after silu's float32."""
import numpy as np
import pytest

from gpu_session import Session, written_everywhere
from oracle import metrics
from rosylnalive_amd.gpu_core import DType, TensorFlags

pytestmark = pytest.mark.gpu

F32, F16 = DType.F32, DType.F16
RO = TensorFlags.READ_ONLY


def _half(r, *s, scale=1.0):
    return (r.standard_normal(s) * scale).astype(np.float16)


@pytest.mark.parametrize("m,n,k", [(1, 4096, 128), (37, 1000, 1024), (64, 16384, 64), (64, 40000, 64), (65, 4097, 128),
                                   (129, 96, 192), (512, 4096, 64)])
def test_gemm_f32_small_tiles(m, n, k):
    r = np.random.default_rng(m + n)
    a, w = _half(r, m, k), _half(r, n, k, scale=0.05)
    s = Session({"a": (F16, (m, k), 0, a.view(np.uint16)), "w": (F16, (n, k), RO, w.view(np.uint16)), "y": (F32, (m, n), 0, None)})
    try:
        y = s.run("gemm_f32", ["y"], a="a", w="w", y="y", m=m, n=n, k=k)["y"]
        assert written_everywhere(y)
        assert metrics.rel_l2(y, a.astype(np.float64) @ w.astype(np.float64).T) < 1e-6
    finally:
        s.close()


@pytest.mark.parametrize("m,n,k,splits", [(17, 1024, 2048, 2), (37, 2048, 2048, 2), (64, 100, 256, 1), (65, 1000, 512, 4),
                                          (256, 1024, 256, 2), (300, 1024, 256, 2), (777, 1024, 256, 4)])
def test_gemm_residual_split_small_tiles(m, n, k, splits):
    r = np.random.default_rng(m + n)
    a, w = _half(r, m, k), _half(r, n, k, scale=0.05)
    s = Session({"a": (F16, (m, k), 0, a.view(np.uint16)), "w": (F16, (n, k), RO, w.view(np.uint16)),
                 "p": (F32, (splits, m, n), 0, None)})
    try:
        p = s.run("gemm_residual_split", ["p"], a="a", w="w", partials="p", m=m, n=n, k=k, splits=splits)["p"]
        ks = k // splits
        for z in range(splits):
            c = slice(z * ks, (z + 1) * ks)
            assert metrics.rel_l2(p.reshape(splits, m, n)[z], a[:, c].astype(np.float64) @ w[:, c].astype(np.float64).T) < 1e-6
    finally:
        s.close()


@pytest.mark.parametrize("m,inter,k", [(1, 3072, 128), (37, 3072, 1024), (64, 6144, 64), (65, 200, 64), (100, 104, 128),
                                       (130, 3000, 64), (300, 6144, 64), (400, 6144, 64), (1500, 3072, 64)])
def test_gemm_swiglu_small_tiles(m, inter, k):
    r = np.random.default_rng(m + inter)
    a, w = _half(r, m, k), _half(r, 2 * inter, k, scale=0.05)
    s = Session({"a": (F16, (m, k), 0, a.view(np.uint16)), "w": (F16, w.shape, RO, w.view(np.uint16)), "y": (F16, (m, inter), 0, None)})
    try:
        y = s.run("gemm_swiglu", ["y"], a="a", w="w", y="y", m=m, inter=inter, k=k, a_shift=0)["y"]
        assert written_everywhere(y)
        g, u = (a.astype(np.float64) @ x.astype(np.float64).T for x in (w[:inter], w[inter:]))
        assert metrics.rel_l2(y.view(np.float16).astype(np.float64), g / (1 + np.exp(-g)) * u) < 3.5e-4
    finally:
        s.close()

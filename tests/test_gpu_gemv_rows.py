"""The one-sequence GEMVs with two rows per wave (4096 rows and up, vectors of 1025 to 2048) and the sizes on either side of
that rule, against float64. Per element, with u = 2^-24: the float32 norm scales every term by 1 + O(20 u), and the dot of K
terms sums K / 64 per lane and six steps across the wave, so |error| <= (K / 64 + 32) u sum|w h|."""
import numpy as np
import pytest

from gpu_session import Session
from oracle import cpuref
from rosylnalive_amd.gpu_core import DType, TensorFlags

pytestmark = pytest.mark.gpu

F32, BF16 = DType.F32, DType.BF16
RO = TensorFlags.READ_ONLY
U = 2.0 ** -24


def bf16(a):
    return cpuref.bf16_narrow(np.asarray(a, np.float32))


def _inputs(rows, k):
    r = np.random.default_rng(rows + k)
    x = (r.standard_normal(k) * 2).astype(np.float32)
    nw = bf16(1 + 0.1 * r.standard_normal(k))
    w = bf16(r.standard_normal((rows, k)) * 0.05)
    h = cpuref.rmsnorm(x[None].astype(np.float64), nw, 1e-6)[0]
    wide = cpuref.bf16_widen(w).astype(np.float64)
    return x, nw, w, wide @ h, (k / 64 + 32) * U * (np.abs(wide) @ np.abs(h))


@pytest.mark.parametrize("n,k", [(4095, 2048), (4096, 2048), (4097, 1032), (4103, 1536), (4100, 2040), (8191, 1024), (4097, 2056)])
def test_gemv_norm_dec_rows(n, k):
    x, nw, w, ref, tol = _inputs(n, k)
    sentinel = np.full(n + 8, 7.0, np.float32)
    s = Session({"x": (F32, (k,), RO, x), "nw": (BF16, (k,), RO, nw), "w": (BF16, (n, k), RO, w),
                 "y": (F32, (n + 8,), 0, sentinel)})
    try:
        s.run_list([("gemv_norm_dec", dict(x="x", norm="nw", w="w", y="y", n=n, k=k, eps=1e-6))], [], reset={"y": sentinel})
        y = s.read("y")
        assert np.all(np.abs(y[:n] - ref) <= tol)
        assert np.all(y[n:] == 7.0)
    finally:
        s.close()


@pytest.mark.parametrize("inter,hidden", [(4095, 1536), (4097, 2048), (4103, 1032), (6144, 1544), (4097, 1024), (4098, 2056)])
def test_gemv_swiglu_dec_rows(inter, hidden):
    x, nw, w, ref, tol = _inputs(2 * inter, hidden)
    sentinel = np.full(inter + 8, 7.0, np.float32)
    s = Session({"x": (F32, (hidden,), RO, x), "nw": (BF16, (hidden,), RO, nw), "w": (BF16, (2 * inter, hidden), RO, w),
                 "y": (F32, (inter + 8,), 0, sentinel)})
    try:
        s.run_list([("gemv_swiglu_dec", dict(x="x", norm="nw", w="w", y="y", inter=inter, hidden=hidden, eps=1e-6))], [],
                   reset={"y": sentinel})
        y = s.read("y")
        g, u = ref[:inter], ref[inter:]
        a = g / (1 + np.exp(-g)) * u
        # |silu'| <= 1.1; the exponential, the division and the two products add at most 8 (1 + |g|) u of the value
        bound = 1.1 * tol[:inter] * np.abs(u) + np.abs(g) * tol[inter:] + 8 * (1 + np.abs(g)) * U * np.abs(a) + 1e-30
        assert np.all(np.abs(y[:inter] - a) <= 1.01 * bound)
        assert np.all(y[inter:] == 7.0)
    finally:
        s.close()

"""argmax_rows at the rows and columns where its workgroup changes: the lowest index of the maximum by '>', also where equal
maxima lie in different threads, zeros of both signs, rows of -inf, and a NaN anywhere in a row (index 0xFFFFFFFF)."""
import numpy as np
import pytest

from gpu_session import Session
from rosylnalive_amd.gpu_core import DType, TensorFlags

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows,cols", [(1, 1), (7, 63), (7, 65), (5000, 512), (6, 513), (600, 1025), (512, 4095), (512, 4096),
                                       (513, 4096), (513, 4100), (5, 32768), (520, 32768), (520, 32769)])
def test_argmax_rows(rows, cols):
    r = np.random.default_rng(rows + cols)
    x = r.integers(-50, 50, (rows, cols)).astype(np.float32)
    x[0] = -np.inf
    x[rows // 2, :] = np.where(r.integers(0, 2, cols), np.float32(0.0), np.float32(-0.0))
    if rows > 4:
        x[3, cols // 2] = x[3, cols - 1] = 1e9
        x[4, r.integers(cols)] = np.nan
    s = Session({"x": (DType.F32, x.shape, TensorFlags.READ_ONLY, x), "y": (DType.U32, (rows,), 0, None)})
    try:
        y = s.run("argmax_rows", ["y"], x="x", y="y", rows=rows, cols=cols)["y"]
        assert np.array_equal(y, np.where(np.isnan(x).any(1), 0xFFFFFFFF, np.argmax(x, 1)).astype(np.uint32))
    finally:
        s.close()

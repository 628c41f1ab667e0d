"""The logical grid that a prepared dispatch of the prefill GEMMs reports is the one that its launch uses: one rule chooses
tile and loop for both. The rows are those at which the rules change sides (CPU)."""
import pytest

from rosylnalive_amd.gpu_core import Arena, ArgBlock, Catalog, DType, HeapPlanner, TensorTable, prepare


def _grid(kernel, tensors, **fields):
    planner = HeapPlanner()
    places = {n: planner.allocate(Arena.ACTIVATIONS, c * DType.SIZE[dt]) for n, (dt, c) in tensors.items()}
    table = TensorTable(planner.build())
    tok = {n: table.add_placed(n, places[n], dt, [c], 0) for n, (dt, c) in tensors.items()}
    return prepare(table.seal(), Catalog.find(kernel).id, ArgBlock.encode(kernel, **tok, **fields))[1]


# 32 heads. Tiles of 128 rows on the direct-to-LDS loop where they mostly fill rounds of 512 (384 and more), else 64 rows where
# those take fewer rounds of 256 (two of them cost more than one of 128)
@pytest.mark.parametrize("m,rows", [(1, 64), (64, 64), (512, 64), (513, 128), (1024, 128), (1408, 128), (1409, 128),
                                    (1500, 128), (1536, 128), (2048, 128), (2049, 128)])
def test_qkv_grid(m, rows):
    F16, BF16, F32 = DType.F16, DType.BF16, DType.F32
    grid = _grid("gemm_qkv_rope",
                 {"h": (F16, m * 64), "w": (F16, 32 * 128 * 64), "q_norm": (BF16, 128), "k_norm": (BF16, 128),
                  "cos_table": (F32, m * 64), "sin_table": (F32, m * 64), "q": (F16, m * 16 * 128),
                  "k_cache": (F16, 8 * 4096 * 128), "v_cache": (F16, 8 * 4096 * 128)},
                 m=m, hidden=64, q_heads=16, kv_heads=8, pos0=0, max_pos=4096, eps=1e-6)
    assert grid == (32, -(-m // rows), 1)

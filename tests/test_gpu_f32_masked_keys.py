"""attention_gqa_causal on the matrix cores, where a key past a query's own could show: the tiles hold such keys with weight
0, and the product 0 * v is a zero of v's sign. Added to a chain that stands at -0 (values whose products underflow) it would
give +0 where the reference, which never sees the key, keeps -0. The tiled kernel (16-byte aligned tensors) equals the
general one (the same tensors one float further) bit for bit there too."""
import numpy as np
import pytest

from test_gpu_f32_mfma import _attention

pytestmark = pytest.mark.gpu

ULP = np.float32(2.0 ** -149)


# 20 and 9 rows: eight waves share a tile; 1030 rows of 64 heads: one wave per tile
@pytest.mark.parametrize("rows,qh,kvh,hd", [(20, 4, 2, 16), (9, 8, 1, 64), (20, 16, 8, 128), (1030, 64, 32, 16)])
def test_values_of_later_keys_leave_a_negative_zero(rows, qh, kvh, hd):
    past = 128
    keys = past + rows
    q, k, v = (np.zeros((n, h * hd), np.float32) for n, h in ((rows, qh), (keys, kvh), (keys, kvh)))
    # scores: 0 in the first key block, one key at 2 in the second, -1 from there on. The output after block 0 is one
    # -2^-149 (key 0), after block 1 exp(-2) of it: -0. The values of the third block carry a weight of exp(-3): those a
    # row owns are -2^-149 up to key past + 4, so its chain there is -0 again, and +2^-149 after.
    q.reshape(rows, qh, hd)[:, :, 0] = np.float32(1.0) / np.float32(hd ** -0.5)
    score = np.full(keys, -1, np.float32)
    score[:64], score[64:128], score[70] = -200, -200, 2
    score[0] = 0
    k.reshape(keys, kvh, hd)[:, :, 0] = score[:, None]
    v[0] = -ULP
    v[past:past + 5] = -ULP
    v[past + 5:] = ULP
    tiled, general = _attention(q, k, v, qh, kvh, hd, past, 0), _attention(q, k, v, qh, kvh, hd, past, 1)
    assert np.array_equal(general[:5].view(np.uint32), np.full((5, qh * hd), 0x80000000, np.uint32))
    assert np.array_equal(tiled.view(np.uint32), general.view(np.uint32))


@pytest.mark.parametrize("rows,past,qh,kvh,hd", [(37, 150, 4, 2, 16), (30, 300, 16, 8, 128), (1030, 5, 64, 32, 16),
                                                 (2800, 70, 6, 3, 16)])
def test_random_denormal_values(rows, past, qh, kvh, hd):
    r = np.random.default_rng(rows + hd)
    keys = past + rows
    q, k = (r.standard_normal((n, h * hd)).astype(np.float32) * 3 for n, h in ((rows, qh), (keys, kvh)))
    v = (r.integers(-2, 3, (keys, kvh * hd)) * np.float64(ULP)).astype(np.float32)
    tiled, general = _attention(q, k, v, qh, kvh, hd, past, 0), _attention(q, k, v, qh, kvh, hd, past, 1)
    assert np.array_equal(tiled.view(np.uint32), general.view(np.uint32))


@pytest.mark.parametrize("hd", [16, 32, 64, 128])
@pytest.mark.parametrize("rows,past,qh,kvh", [(1, 0, 4, 2), (1, 9, 16, 8), (1, 10, 16, 8), (1, 12, 6, 2), (1, 13, 4, 1),
                                              (3, 7, 16, 8), (3, 8, 16, 8), (12, 0, 16, 8), (13, 0, 4, 4), (9, 0, 512, 128),
                                              (6, 0, 512, 256)])
def test_few_keys(rows, past, qh, kvh, hd):
    """Either side of the counts up to which the general kernel takes aligned tensors too."""
    r = np.random.default_rng(rows + past + hd)
    q, k, v = (r.standard_normal((n, h * hd)).astype(np.float32) for n, h in ((rows, qh), (past + rows, kvh), (past + rows, kvh)))
    tiled, general = _attention(q, k, v, qh, kvh, hd, past, 0), _attention(q, k, v, qh, kvh, hd, past, 1)
    assert np.array_equal(tiled.view(np.uint32), general.view(np.uint32))

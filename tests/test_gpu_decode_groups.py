"""GPU: one-row attention at the edges of its key chunks, for every head
dimension and for whole, partial and several groups of query heads; the bound is
test_gpu_prefill_split's.
"""
import numpy as np
import pytest

from test_gpu_prefill_split import attend, check, inputs

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("d", [4, 8, 16, 32, 64, 128, 256])
@pytest.mark.parametrize("group", [1, 2, 3, 4, 5, 8, 9])
def test_groups(dev, group, d):
    chunk = {4: 512, 8: 512}.get(d, 8 * 1024 // d)
    for keys, window in ((1, None), (chunk - 1, None), (chunk, None), (chunk + 1, None), (3 * chunk + 7, chunk + 2)):
        q, k, v = inputs(keys + group, 1, keys, 2 * group, 2, d)
        got = attend(dev, q, k, v, 1, keys, 2 * group, 2, d, causal=True, window_size=window)
        check(got, q, k, v, 1, keys, 2 * group, 2, d, True, window)


@pytest.mark.parametrize("group", [1, 2, 4])
@pytest.mark.parametrize("d", [16, 128])
def test_chunks_of_twice_the_steps(dev, d, group):
    from magnetar_hip import ops
    hkv, keys = 16, 8 * 1024 // d * 4 + 3
    batch = 16 * 256 // (hkv * 5) + 1
    q, k, v = inputs(d, batch, batch * keys, hkv * group, hkv, d)
    p = ops.attention_params(1, keys, hkv * group, d, kv_head_count=hkv, causal=True, batch=batch)
    got = ops.attention(dev, dev.upload(q), dev.upload(k), dev.upload(v), p).numpy()
    for b in (0, batch - 1):
        rows = slice(b * keys, (b + 1) * keys)
        check(got[b:b + 1], q[b:b + 1], k[rows], v[rows], 1, keys, hkv * group, hkv, d, True)


@pytest.mark.parametrize("d", [8, 64, 128])
def test_values_that_are_not_finite(dev, d):
    """Rows and columns that do not meet them are as they are without."""
    q, k, v = inputs(d, 1, 700, 8, 2, d)
    plain = attend(dev, q, k, v, 1, 700, 8, 2, d, causal=True)
    v[650, 1], v[3, d + 2] = np.inf, np.nan
    got = attend(dev, q, k, v, 1, 700, 8, 2, d, causal=True)
    met = np.zeros((8, d), bool)
    met[:4, 1] = met[4:, 2] = True
    assert np.all(got.reshape(8, d)[:4, 1] == np.inf) and np.all(np.isnan(got.reshape(8, d)[4:, 2]))
    assert np.array_equal(got.reshape(8, d)[~met], plain.reshape(8, d)[~met])
    k[:] = 0.0
    v = np.full_like(v, 3e38)
    assert np.all(np.abs(attend(dev, q, k, v, 1, 700, 8, 2, d, causal=True) / np.float32(3e38) - 1) < 1e-6)

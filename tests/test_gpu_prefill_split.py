"""GPU: prompt attention on the split bf16 matrix products at the edges of its
tiles, head dimensions and operand ranges, replayed, and in a capture that has
no room for its key chunks.

Bound: a score is off by at most (d + 16) u |q| |k| scale (u = 2^-24: the f32
sum of d products and the roundings of q's scaling, the split and the
exponent), which moves every weight by that much relative to it and the output
by twice the largest such error; the weighted mean itself adds (keys + 64) u.
Both scale with the largest admitted |v| of the column.
"""
import numpy as np
import pytest

from conftest import bits

pytestmark = pytest.mark.gpu

U = 2.0 ** -24


def inputs(seed, s, kv, h, hkv, d):
    rng = np.random.default_rng(seed)
    return [rng.standard_normal((r, c)).astype(np.float32) for r, c in ((s, h * d), (kv, hkv * d), (kv, hkv * d))]


def attend(dev, q, k, v, s, kv, h, hkv, d, **kw):
    from magnetar_hip import ops
    p = ops.attention_params(s, kv, h, d, kv_head_count=hkv, **kw)
    return ops.attention(dev, dev.upload(q), dev.upload(k), dev.upload(v), p).numpy()


def check(got, q, k, v, s, kv, h, hkv, d, causal=False, window_size=None, rows=None):
    """Every (row, head) against float64; rows: the ones with finite admitted values."""
    pos, scale = np.arange(kv), 1.0 / np.sqrt(np.float64(d))
    for i in range(s) if rows is None else rows:
        at = kv - s + i
        admitted = (pos <= at) if causal else np.full(kv, True)
        if window_size:
            admitted &= pos > at - window_size
        for head in range(h):
            g = head // (h // hkv)
            Q = q[i, head * d:(head + 1) * d].astype(np.float64)
            K = k[admitted, g * d:(g + 1) * d].astype(np.float64)
            V = v[admitted, g * d:(g + 1) * d].astype(np.float64)
            x = K @ Q * scale
            w = np.exp(x - x.max())
            want = (w / w.sum()) @ V
            score_error = (d + 16) * U * (np.abs(K) @ np.abs(Q)).max() * scale
            bound = (2 * score_error + (len(V) + 64) * U) * np.abs(V).max(axis=0)
            err = np.abs(got[i, head * d:(head + 1) * d] - want)
            assert np.all(err <= bound), (i, head, (err / bound).max())


SHAPES = [  # s, kv, h, hkv, causal, window
    (1, 1, 2, 1, True, None), (31, 31, 3, 3, True, None), (32, 33, 2, 2, False, None), (33, 64, 4, 2, True, 7),
    (255, 300, 2, 1, True, None), (257, 257, 2, 2, True, 40), (5, 1030, 4, 2, True, None), (40, 700, 2, 2, True, 300)]


@pytest.mark.parametrize("d", [32, 64, 80, 96, 112, 128])
@pytest.mark.parametrize("s,kv,h,hkv,causal,window", SHAPES)
def test_edges_of_tiles(dev, s, kv, h, hkv, causal, window, d):
    q, k, v = inputs(s + d, s, kv, h, hkv, d)
    got = attend(dev, q, k, v, s, kv, h, hkv, d, causal=causal, window_size=window)
    check(got, q, k, v, s, kv, h, hkv, d, causal, window)


@pytest.mark.parametrize("d", [32, 64])
@pytest.mark.parametrize("window", [None, 50])
def test_128_queries_have_the_bits_of_129(dev, d, window):
    """Workgroups of four waves (more than one round of them) and of eight: the
    same queries, the same bits."""
    from magnetar_hip import ops
    kv, h, hkv, batch = 200, 4, 2, 65
    q, k, v = inputs(d, 129, kv, h, hkv, d)
    want = attend(dev, q, k, v, 129, kv, h, hkv, d, causal=True, window_size=window)[1:]
    p = ops.attention_params(128, kv, h, d, kv_head_count=hkv, causal=True, window_size=window, batch=batch)
    many = [dev.upload(np.tile(x, (batch, 1))) for x in (q[1:], k, v)]
    got = ops.attention(dev, *many, p).numpy().reshape(batch, 128, h * d)
    for one in (attend(dev, q[1:], k, v, 128, kv, h, hkv, d, causal=True, window_size=window), got[0], got[64]):
        assert np.array_equal(bits(one), bits(want))
    check(got[33], q[1:], k, v, 128, kv, h, hkv, d, True, window)


@pytest.mark.parametrize("s,kv", [(1, 33), (7, 420), (31, 64), (127, 300)])
def test_batches_of_few_queries(dev, s, kv):
    """Four waves a workgroup, a batch its separate calls bit for bit."""
    from magnetar_hip import ops
    d, h, hkv, batch = 32, 16, 4, 17
    q, k, v = inputs(s, s, kv, h, hkv, d)
    p = ops.attention_params(s, kv, h, d, kv_head_count=hkv, causal=True, batch=batch)
    got = ops.attention(dev, *[dev.upload(np.tile(x, (batch, 1))) for x in (q, k, v)], p).numpy().reshape(batch, s, h * d)
    one = attend(dev, q, k, v, s, kv, h, hkv, d, causal=True)
    check(one, q, k, v, s, kv, h, hkv, d, True)
    assert all(np.array_equal(bits(got[b]), bits(one)) for b in range(batch))


@pytest.mark.parametrize("d", [32, 96, 128])
def test_a_batch_is_its_sequences(dev, d):
    from magnetar_hip import ops
    s, kv, h = 70, 300, 4
    q, k, v = inputs(d, 3 * s, 3 * kv, h, 2, d)
    p = ops.attention_params(s, kv, h, d, kv_head_count=2, causal=True, batch=3)
    got = ops.attention(dev, dev.upload(q), dev.upload(k), dev.upload(v), p).numpy()
    for b in range(3):
        rs, rk = slice(b * s, (b + 1) * s), slice(b * kv, (b + 1) * kv)
        one = attend(dev, q[rs], k[rk], v[rk], s, kv, h, 2, d, causal=True)
        assert np.array_equal(bits(got[rs]), bits(one))


@pytest.mark.parametrize("d", [64, 80, 112, 128])
@pytest.mark.parametrize("what", ["q 2^70", "k 2^65", "v 3e38", "v 1e-40", "v scale 1e-25", "one v 1e-30", "v inf"])
def test_operands_outside_the_split(dev, d, what):
    s, kv, h, hkv = 100, 300, 4, 2
    q, k, v = inputs(d, s, kv, h, hkv, d)
    rows = None
    if what == "q 2^70":
        q, k = q * np.float32(2.0 ** 70), k * np.float32(2.0 ** -70)
    elif what == "k 2^65":
        q, k = q * np.float32(2.0 ** -65), k * np.float32(2.0 ** 65)
    elif what == "v 3e38":
        v = np.sign(v) * np.float32(3e38)
    elif what == "v 1e-40":
        v[50:60] = 1e-40
    elif what == "v scale 1e-25":
        v *= np.float32(1e-25)
    elif what == "one v 1e-30":
        v[:, 3] = 1e-30
    else:
        v[210, 5] = np.inf  # first admitted by query 10, and 9 rows of its wave mask it
        rows = range(10)
    got = attend(dev, q, k, v, s, kv, h, hkv, d, causal=True)
    check(got, q, k, v, s, kv, h, hkv, d, True, rows=rows)
    if what == "v inf":
        assert np.all(np.isinf(got[10:, 5]) & np.isinf(got[10:, d + 5])) and np.all(np.isfinite(got[:, :5]))


@pytest.mark.parametrize("d", [32, 64, 80, 112, 128])
@pytest.mark.parametrize("kv", [270, 1000])  # whole, and in key chunks
def test_what_lies_outside_moves_its_own_queries_only(dev, d, kv):
    """A key beyond 2^60 moves the queries that admit it, a query that one, and a
    tiny value among ordinary ones no output."""
    s, h, hkv = 260 if kv == 270 else 40, 4, 2
    q, k, v = inputs(d + kv, s, kv, h, hkv, d)
    want = bits(attend(dev, q, k, v, s, kv, h, hkv, d, causal=True))
    at = kv - s + s // 2  # first admitted by query s // 2
    far = k.copy()
    far[at] = np.float32(2.0 ** 61)
    got = bits(attend(dev, q, far, v, s, kv, h, hkv, d, causal=True))
    assert np.array_equal(got[:s // 2], want[:s // 2]) and not np.array_equal(got[s // 2:], want[s // 2:])
    big = q.copy()
    big[s // 3] *= np.float32(2.0 ** 61)
    got = bits(attend(dev, big, k, v, s, kv, h, hkv, d, causal=True))
    others = np.arange(s) != s // 3
    assert np.array_equal(got[others], want[others])
    got = []
    for value in (0.0, 1e-30, 1e-44):
        few = v.copy()
        few[5::17, ::3] = value
        got.append(bits(attend(dev, q, k, few, s, kv, h, hkv, d, causal=True)))
    assert np.array_equal(got[0], got[1]) and np.array_equal(got[0], got[2])


@pytest.mark.parametrize("d", [32, 80, 128])
@pytest.mark.parametrize("kv", [270, 1000])
def test_columns_of_tiny_values(dev, d, kv):
    """Each column at its own scale, down to values that vanish when scaled."""
    s, h, hkv = 40, 4, 2
    q, k, v = inputs(d, s, kv, h, hkv, d)
    v *= (2.0 ** -np.linspace(60.0, 124.0, hkv * d)).astype(np.float32)
    check(attend(dev, q, k, v, s, kv, h, hkv, d, causal=True), q, k, v, s, kv, h, hkv, d, True)
    v[:, 3] = np.float32(1e-43)  # a denormal's mean is itself, to a few of the least f32
    got = attend(dev, q, k, v, s, kv, h, hkv, d, causal=True)
    assert np.all(np.abs(got[:, [3, 3 + d]] - np.float32(1e-43)) <= 64 * 2.0 ** -149)


@pytest.mark.parametrize("d", [80, 96, 128])
def test_a_replayed_row_has_the_bits_of_the_call(dev, d):
    from magnetar_hip import ops
    from magnetar_hip.device import ADVANCE_KEY_COUNT
    q, k, v = inputs(d, 1, 2000, 4, 2, d)
    dq, dk, dv = dev.upload(q), dev.upload(k), dev.upload(v)
    def call(keys, out=None):
        p = ops.attention_params(1, 2000, 4, d, kv_head_count=2, causal=True, key_count=keys)
        return ops.attention(dev, dq, dk, dv, p, out)
    want = {keys: call(keys).numpy() for keys in (300, 301, 1999)}
    out = dev.empty((1, 4 * d))
    dev.capture_begin(ADVANCE_KEY_COUNT)
    call(300, out)
    graph = dev.capture_end()
    for keys in (300, 1999, 301, 1999):
        graph.launch(keys - 300)
        assert np.array_equal(bits(out.numpy()), bits(want[keys]))


def test_a_cold_capture_of_attention():
    import magnetar_hip
    from magnetar_hip import ops
    q, k, v = inputs(1, 3, 2000, 4, 2, 96)
    fresh = magnetar_hip.Device(0)
    dq, dk, dv, out = fresh.upload(q), fresh.upload(k), fresh.upload(v), fresh.empty((3, 4 * 96))
    p = ops.attention_params(3, 2000, 4, 96, kv_head_count=2, causal=True)
    fresh.capture_begin(0)
    ops.attention(fresh, dq, dk, dv, p, out)
    graph = fresh.capture_end()
    for _ in range(2):
        graph.launch(0)
        check(out.numpy(), q, k, v, 3, 2000, 4, 2, 96, True)


@pytest.mark.parametrize("d", [32, 80, 128])
@pytest.mark.parametrize("kv", [1, 33, 54])
def test_nothing_is_read_past_the_last_key(dev, d, kv):
    """What lies behind K and V (the next rows of the same allocation, 31 at
    most of a last tile of 32 keys) leaves the bits alone, NaN or not."""
    import magnetar_hip
    from magnetar_hip import ops
    q, k, v = inputs(kv, kv, kv + 32, 2, 2, d)
    p = ops.attention_params(kv, kv, 2, d, kv_head_count=2, causal=True)
    got = []
    for behind in (0.0, np.nan):
        k[kv:] = v[kv:] = behind
        dk, dv = dev.upload(k), dev.upload(v)
        views = [magnetar_hip.DeviceArray(dev, x.ptr, (kv, 2 * d), x.dtype, owned=False) for x in (dk, dv)]
        got.append(ops.attention(dev, dev.upload(q), *views, p).numpy())
    assert np.array_equal(bits(got[0]), bits(got[1]))

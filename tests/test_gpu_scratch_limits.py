"""GPU: products whose fastest plan wants more scratch than an entry point has,
where the plans of the f32 matrix instructions wanted less: they are taken, on
a plan that fits. |C - C64| <= (k + 8) u (|A| |B|), u = 2^-24 (Higham, Accuracy
and Stability of Numerical Algorithms, eq. 3.5)."""
import ctypes

import numpy as np
import pytest

from conftest import bits

pytestmark = pytest.mark.gpu

U = 2.0 ** -24


# A small ragged row, a panel, a row stored as a column and tiles, all of whose
# fastest plans take partial sums where the f32 kernels' took none.
@pytest.mark.parametrize("m,k,n,ta", [(1, 64, 10, False), (20, 480, 640, False), (1, 480, 64, True), (192, 3072, 5120, False)])
def test_a_cold_capture_of_a_product(m, k, n, ta):
    import magnetar_hip
    from magnetar_hip import ops
    rng = np.random.default_rng(m)
    a = rng.standard_normal((m, k)).astype(np.float32)
    b = rng.standard_normal((k, n)).astype(np.float32)
    fresh = magnetar_hip.Device(0)
    da, db, out = fresh.upload(a.reshape(k, m) if ta else a), fresh.upload(b), fresh.empty((m, n))
    fresh.capture_begin(0)
    ops.matmul(fresh, da, db, ta, False, out=out)
    graph = fresh.capture_end()
    wide = b.astype(np.float64)
    bound = (k + 8) * U * (np.abs(a).astype(np.float64) @ np.abs(wide))
    for _ in range(2):
        graph.launch(0)
        assert np.all(np.abs(out.numpy() - a.astype(np.float64) @ wide) <= bound)


# The same, a product whose partial sums are stream-K's, and prompts in key
# chunks: a capture takes the eager call's plan, so its replays have its bits.
CALLS = [("matmul", (1, 64, 10, False)), ("matmul", (20, 480, 640, False)), ("matmul", (1, 480, 64, True)),
         ("matmul", (192, 3072, 5120, False)), ("matmul", (5, 500, 333, False)), ("matmul", (31, 500, 1030, False)),
         ("attention", (3, 2000, 4, 2, 96)), ("attention", (300, 1000, 8, 8, 80)), ("attention", (40, 600, 2, 1, 32))]


def call_of(kind, shape):
    """make(device) -> (run, out): the call on that device, its inputs the same on every one."""
    from magnetar_hip import ops
    rng = np.random.default_rng(sum(shape))
    normal = lambda *s: rng.standard_normal(s).astype(np.float32)
    if kind == "matmul":
        m, k, n, ta = shape
        host = [normal(k, m) if ta else normal(m, k), normal(k, n)]
        def make(device):
            da, db, out = device.upload(host[0]), device.upload(host[1]), device.empty((m, n))
            return (lambda: ops.matmul(device, da, db, ta, False, out=out)), out
        return make
    s, kv, h, hkv, d = shape
    host = [normal(s, h * d), normal(kv, hkv * d), normal(kv, hkv * d)]
    def make(device):
        q, k, v, out = *map(device.upload, host), device.empty((s, h * d))
        p = ops.attention_params(s, kv, h, d, kv_head_count=hkv, causal=True)
        return (lambda: ops.attention(device, q, k, v, p, out)), out
    return make


@pytest.mark.parametrize("kind,shape", CALLS)
def test_a_cold_capture_has_the_eager_bits(dev, kind, shape):
    import magnetar_hip
    make = call_of(kind, shape)
    run, out = make(dev)
    run()
    want = bits(out.numpy())
    fresh = magnetar_hip.Device(0)
    run, out = make(fresh)
    fresh.capture_begin(0)
    run()
    graph = fresh.capture_end()
    for _ in range(2):
        fresh.zeros(out.shape)  # (eager work between replays)
        graph.launch(0)
        assert np.array_equal(bits(out.numpy()), want)


def test_growing_for_a_capture_leaves_earlier_launches_their_scratch():
    """A workspace that grows while recording: the launches recorded before it,
    in the same capture and in a live graph, keep theirs."""
    import magnetar_hip
    fresh, other = magnetar_hip.Device(0), magnetar_hip.Device(0)
    calls = [call_of(*CALLS[i]) for i in (0, 1, 3, 7)]
    runs, outs = zip(*(make(fresh) for make in calls))
    wants = []
    for make in calls:
        run, out = make(other)
        run()
        wants.append(bits(out.numpy()))
    graphs = []
    for some in ((0,), (0, 1), (0, 1, 2, 3)):
        fresh.capture_begin(0)
        for i in some:
            runs[i]()
        graphs.append((some, fresh.capture_end()))
    fresh.capture_begin(0)
    runs[2]()
    fresh.capture_abort()
    for some, graph in graphs * 2:
        graph.launch(0)
        for i in some:
            assert np.array_equal(bits(outs[i].numpy()), wants[i])
    for _, graph in graphs:
        graph.close()
    runs[3]()
    assert np.array_equal(bits(outs[3].numpy()), wants[3])


def test_a_product_the_fixed_scratch_took_is_taken(dev):
    """The fastest tiles of 3392 x 5056 x 5952 want 162 MB of partial sums."""
    from magnetar_hip import _lib, ops
    m, k, n = 3392, 5056, 5952
    rng = np.random.default_rng(0)
    a, b = dev.upload(rng.standard_normal((m, k)).astype(np.float32)), dev.upload(rng.standard_normal((k, n)).astype(np.float32))
    out = dev.empty((m, n))
    p = lambda x: ctypes.c_void_p(x.ptr)
    assert _lib.lib().mhip_matmul_f32_noalloc(dev.ctx, p(a), p(b), p(out), m, k, n, 0, 0, None, 0) == 0
    assert np.array_equal(bits(out.numpy()), bits(ops.matmul(dev, a, b).numpy()))

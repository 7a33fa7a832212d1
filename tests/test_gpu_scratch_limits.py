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

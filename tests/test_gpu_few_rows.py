"""GPU: the few-row products (csrc/few_rows.hpp) and the softmax of wide or
ragged rows at the edges of their ranges.

Products: |C - C64| <= (k + 8) u (|A| |B|) entry by entry, u = 2^-24 (Higham,
Accuracy and Stability of Numerical Algorithms, eq. 3.5, with 8 u for a split
product's dropped terms and an addend's rounding), every addend form the bits
of the product followed by the addition, and a compact weight the bits of its
f32 widening. Softmax: (2 |x - M| + 32) u of each entry: the rounding of the two differences
under the exponentials, and some thirty more (exponentials, the scaling, a
sum of up to 48 terms a thread and then in pairs).
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def check_products(dev, m, k, n, tb, path, poison=None):
    from magnetar_hip import ops
    assert ops.matmul_plan(dev, m, k, n, False, tb)["path"] == path
    rng = np.random.default_rng(1000 * m + n)
    a = rng.standard_normal((m, k)).astype(np.float32)
    bits = (rng.standard_normal((n, k) if tb else (k, n)).astype(np.float32).view(np.uint32) >> 16).astype(np.uint16)
    if poison is not None:
        a[m - 1, k // 2] = poison
        bits[k // 3 if not tb else n // 2, n // 2 if not tb else k // 3] = 0xFF80  # -inf
    b = (bits.astype(np.uint32) << 16).view(np.float32)
    da, db, dh = dev.upload(a), dev.upload(b), dev.upload(bits)
    plain = ops.matmul(dev, da, db, False, tb)
    got = plain.numpy()
    wide = b.T if tb else b
    with np.errstate(all="ignore"):
        exact = a.astype(np.float64) @ wide.astype(np.float64)
        scale = np.abs(a).astype(np.float64) @ np.abs(wide).astype(np.float64)
        fine = scale < 3e38  # no partial sum overflows
        assert np.all(np.abs(got - exact)[fine] <= (k + 8) * 2.0 ** -24 * scale[fine])
        special = ~np.isfinite(scale)
        assert np.array_equal(np.isnan(got[special]), np.isnan(exact[special]))
        inf = np.isinf(exact)
        assert np.array_equal(got[inf], exact[inf].astype(np.float32))
    assert np.array_equal(ops.matmul_bf16w(dev, da, dh, False, tb).numpy().view(np.uint32), got.view(np.uint32))
    bias = dev.upload(rng.standard_normal(n).astype(np.float32))
    res = dev.upload(rng.standard_normal((m, n)).astype(np.float32))
    for mode, add, want in ((1, bias, ops.bias_add(dev, plain, bias)), (2, res, ops.add(dev, plain, res))):
        fused = ops.matmul(dev, da, db, False, tb, add, mode).numpy()
        assert np.array_equal(fused.view(np.uint32), want.numpy().view(np.uint32))


@pytest.mark.parametrize("m", [1, 2, 5, 8])
@pytest.mark.parametrize("k,n", [(1, 1), (31, 255), (64, 33), (65, 33), (4096, 257), (1030, 1029), (300, 50257)])
def test_ragged_gemv(dev, m, k, n):
    check_products(dev, m, k, n, False, "gemv_ragged")


@pytest.mark.parametrize("m", [1, 2, 3, 7, 8])
@pytest.mark.parametrize("k,n", [(8, 1), (512, 7), (520, 4097), (1024, 8191), (4096, 259)])
def test_row_dots(dev, m, k, n):
    check_products(dev, m, k, n, True, "row_dots")


@pytest.mark.parametrize("m,k,n,path", [(1, 32, 32001, "row_dots"), (3, 32, 8193, "tiles"), (8, 128, 8193, "tiles"),
                                        (8, 128, 8192, "row_dots"), (8, 16392, 130, "tiles"), (8, 16384, 130, "row_dots"),
                                        (4, 32768, 128, "row_dots"), (5, 32776, 33, "tiles")])
def test_row_dots_where_they_are_faster(dev, m, k, n, path):
    check_products(dev, m, k, n, True, path)


@pytest.mark.parametrize("m,k,n", [(9, 1, 2), (9, 15, 30), (10, 257, 258), (17, 1000, 510), (31, 4100, 514),
                                   (32, 4096, 11008), (25, 2050, 4098), (12, 33, 32),
                                   (30, 65, 4094)])
def test_row_panel(dev, m, k, n):
    check_products(dev, m, k, n, False, "row_panel")


# 64 and more partial results of a long k, whole vectors of them and not.
@pytest.mark.parametrize("m,k,n,path", [(17, 9300, 66, "row_panel"), (9, 9500, 64, "row_panel"), (32, 65536, 130, "row_panel"),
                                        (3, 20000, 7, "gemv_ragged"), (8, 2049, 253, "gemv_ragged")])
def test_sums_of_many_slices(dev, m, k, n, path):
    from magnetar_hip import ops
    assert ops.matmul_plan(dev, m, k, n)["splits"] >= 64
    check_products(dev, m, k, n, False, path)


@pytest.mark.parametrize("poison", [np.inf, np.nan, -3.4e38, 1e-44])
@pytest.mark.parametrize("m,k,n,tb,path", [(9, 100, 258, False, "row_panel"), (31, 1030, 600, False, "row_panel"),
                                           (2, 520, 100, True, "row_dots"), (4, 77, 99, False, "gemv_ragged")])
def test_values_outside_the_split(dev, m, k, n, tb, path, poison):
    check_products(dev, m, k, n, tb, path, poison)


@pytest.mark.parametrize("m,k,n", [(9, 1, 2), (17, 33, 510), (12, 54, 258)])
@pytest.mark.parametrize("compact", [False, True])
def test_row_panel_reads_nothing_past_b(dev, m, k, n, compact):
    """What lies behind B (here the next rows of the same allocation, 15 at
    most of a last step of 16 k) leaves the bits alone, NaN or not: one read
    would send the columns to the f32 MFMA's sums."""
    import magnetar_hip
    from magnetar_hip import ops
    rng = np.random.default_rng(k)
    a = dev.upload(rng.standard_normal((m, k)).astype(np.float32))
    full = rng.standard_normal((k + 16, n)).astype(np.float32)
    got = []
    for behind in (0.0, np.nan):
        full[k:] = behind
        d = dev.upload((full.view(np.uint32) >> 16).astype(np.uint16) if compact else full)
        b = magnetar_hip.DeviceArray(dev, d.ptr, (k, n), d.dtype, owned=False)
        got.append((ops.matmul_bf16w if compact else ops.matmul)(dev, a, b).numpy().view(np.uint32))
    assert np.array_equal(got[0], got[1])


WIDTHS = [1, 63, 255, 1023, 1025, 4095, 4097, 16383, 16385, 16388, 32768, 32772, 49151, 49153, 65536, 65540, 70001,
          128000]


# Around the edges of the rows that a wave, several of it in a workgroup, or a
# small workgroup holds.
SHORT = [2, 65, 257, 509, 513, 2047, 2049, 8191, 8193]


@pytest.mark.parametrize("cols,rows", [(c, 3) for c in WIDTHS] + [(c, 9) for c in SHORT])
def test_softmax_of_wide_and_ragged_rows(dev, cols, rows):
    from magnetar_hip import ops
    rng = np.random.default_rng(cols)
    x = (4 * rng.standard_normal((rows, cols))).astype(np.float32)
    if cols > 2:
        x[1, : cols // 2] = -np.inf
        x[2, cols - 1] = 80.0
    d = dev.upload(x)
    got = ops.softmax_rows(dev, d).numpy()
    assert dev.check_flags() == 0
    e = np.exp(x.astype(np.float64) - x.max(1, keepdims=True))
    want = e / e.sum(1, keepdims=True)
    with np.errstate(all="ignore"):
        far = np.where(want > 0, x.max(1, keepdims=True).astype(np.float64) - x, 0)
    assert np.all(np.abs(got - want) <= (2 * far + 32) * 2.0 ** -24 * want + 1e-37)
    ops.softmax_rows(dev, d, out=d)  # in place
    assert np.array_equal(d.numpy().view(np.uint32), got.view(np.uint32))


@pytest.mark.parametrize("cols", WIDTHS[3:] + SHORT[1:])
def test_softmax_keeps_nan_and_flags_rows_without_a_finite_entry(dev, cols):
    import magnetar_hip
    from magnetar_hip import ops
    x = np.full((3, cols), -np.inf, np.float32)
    x[0] = 1.0
    x[0, 7] = np.nan
    x[1, 0] = np.nan  # a finite entry far from the NaN
    x[1, cols - 1] = 2.0
    x[2, 5] = 3.0
    got = ops.softmax_rows(dev, dev.upload(x)).numpy()
    assert dev.check_flags() == 0
    assert np.all(np.isnan(got[:2])) and got[2, 5] == 1.0 and np.count_nonzero(got[2]) == 1
    x[1] = -np.inf
    x[1, 3] = np.nan
    ops.softmax_rows(dev, dev.upload(x))
    with pytest.raises(magnetar_hip.MagnetarHipError):
        dev.check_flags()

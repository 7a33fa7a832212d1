"""GPU: the f32 products summed as bf16 plane products (csrc/split_tile.hpp),
one shape per tile configuration, at the values where the split does not hold:
infinities, NaN, the largest and the smallest f32, and rows so small that
their planes would underflow. The sums that these may matter to, and no other,
are summed again with the f32 MFMA.

Bound, entry by entry: |C - C64| <= (k + 8) u (|A| |B|) with u = 2^-24, the
forward-error bound of any order of f32 additions (Higham, Accuracy and
Stability of Numerical Algorithms, eq. 3.5) plus 8 u for the split (its planes
are exact, its dropped products a2 b3 + a3 b2 + a3 b3 below 1.01 u of |A| |B|:
|x2| <= 2^-8 |x|, |x3| <= 2^-17 |x|; six roundings a product where there are
few) and the first-order bound's remainder. Entries that are not finite in f64 rounded to
f32 are compared exactly.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# (m, k, n, tile): ragged edges and a k that ends inside a stage.
SHAPES = [(70, 90, 70), (64, 200, 2050), (2000, 72, 2030), (3190, 530, 3970), (4000, 72, 4060), (4000, 7, 4060)]


def check(got, a, b):
    k = a.shape[1]
    with np.errstate(all="ignore"):
        exact = a.astype(np.float64) @ b.astype(np.float64)
        as_f32 = exact.astype(np.float32)
        scale = np.abs(a).astype(np.float64) @ np.abs(b).astype(np.float64)
        fine = np.isfinite(as_f32) & (scale < 3e38)
        bound = (k + 8) * 2.0 ** -24 * scale[fine] + 2.0 ** -140
        err = np.abs(got[fine] - exact[fine])
    assert np.all(err <= bound), f"{np.max(err / bound):.2f} of the bound"
    # Entries whose terms hold an infinity or NaN (not mere overflow of a sum).
    special = ~np.isfinite(scale)
    assert np.array_equal(np.isnan(got[special]), np.isnan(as_f32[special]))
    inf = special & np.isinf(as_f32)
    assert np.array_equal(got[inf], as_f32[inf])
    return int(fine.sum()), int(special.sum())


def operands(m, k, n, seed):
    rng = np.random.default_rng(seed)
    return (rng.standard_normal((m, k)).astype(np.float32),
            (0.05 * rng.standard_normal((k, n))).astype(np.float32))


def variants(dev, a, b):
    """The product with the operands stored as they are and transposed."""
    from magnetar_hip import ops
    out = [ops.matmul(dev, dev.upload(a), dev.upload(b)).numpy()]
    at, bt = np.ascontiguousarray(a.T), np.ascontiguousarray(b.T)
    out.append(ops.matmul(dev, dev.upload(at), dev.upload(bt), True, True).numpy())
    assert np.array_equal(out[0].view(np.uint32), out[1].view(np.uint32))
    return out[0]


def test_the_shapes_cover_every_configuration(dev):
    from magnetar_hip import ops
    plans = [ops.matmul_plan(dev, *shape) for shape in SHAPES]
    assert {(p["tile"][0], p["waves"]) for p in plans} == {(64, 8), (128, 4), (128, 8), (256, 8)}, plans


@pytest.mark.parametrize("m,k,n", SHAPES)
def test_finite_values_meet_the_f32_bound(dev, m, k, n):
    a, b = operands(m, k, n, m + n)
    a[m // 2] = 0.0
    a[:, k // 3] *= np.float32(2.0 ** 60)   # wide ranges inside one sum
    b[k // 3] *= np.float32(2.0 ** -60)
    check(variants(dev, a, b), a, b)


@pytest.mark.parametrize("m,k,n", SHAPES)
@pytest.mark.parametrize("value", [np.inf, -np.inf, np.nan, 3.4028235e38, -3.4028235e38, 1e-45, 2e-38])
def test_values_outside_the_split(dev, m, k, n, value):
    """One such value in A, one in B (in other tiles where there are several)."""
    a, b = operands(m, k, n, m + 7)
    a[m - 1, k - 1] = value
    b[0, n // 2] = value
    finite, special = check(variants(dev, a, b), a, b)
    assert finite > 0
    assert (special > 0) == (not np.isfinite(np.float32(value)))


@pytest.mark.parametrize("m,k,n", SHAPES)
@pytest.mark.parametrize("down", [-100, -108, -120])
def test_small_rows_keep_their_precision(dev, m, k, n, down):
    """Rows of A at 2^down against columns of B at 2^90: their products are
    ordinary numbers and as exact as any."""
    a, b = operands(m, k, n, m + 13)
    a[::3] *= np.float32(2.0 ** down)
    b *= np.float32(2.0 ** 90)
    check(variants(dev, a, b), a, b)


@pytest.mark.parametrize("m,k,n", SHAPES)
def test_compact_weights_give_the_f32_bits(dev, m, k, n):
    """Also where a tile is summed again: a bf16 infinity, and odd widths."""
    from magnetar_hip import ops
    for special in (False, True):
        a, b = operands(m, k, n - 1, m + 17)
        bits = (b.view(np.uint32) >> 16).astype(np.uint16)
        if special:
            bits[k // 2, 1] = 0x7F80
        wide = (bits.astype(np.uint32) << 16).view(np.float32)
        da = dev.upload(a)
        want = ops.matmul(dev, da, dev.upload(wide)).numpy()
        got = ops.matmul_bf16w(dev, da, dev.upload(bits)).numpy()
        assert np.array_equal(got.view(np.uint32), want.view(np.uint32))
        check(want, a, wide)


# One shape per tile configuration, k split over workgroups, stream-K, row panels.
PLACES = SHAPES[:5] + [(509, 1100, 1500), (192, 3072, 5120), (512, 1024, 11008), (20, 480, 640), (31, 200, 258)]


@pytest.mark.parametrize("m,k,n", PLACES)
@pytest.mark.parametrize("value", [np.inf, np.nan, 3.4e38, 1e-44])
def test_a_value_moves_its_own_row_and_column_only(dev, m, k, n, value):
    """The other entries keep the bits they have without it."""
    from magnetar_hip import ops
    a, b = operands(m, k, n, m + 23)
    want = ops.matmul(dev, dev.upload(a), dev.upload(b)).numpy().view(np.uint32)
    row, col = m // 3, n // 2
    a[row, k // 2] = b[k // 3, col] = value
    got = ops.matmul(dev, dev.upload(a), dev.upload(b)).numpy().view(np.uint32)
    others = np.ones((m, n), bool)
    others[row, :] = others[:, col] = False
    assert np.array_equal(got[others], want[others])


@pytest.mark.parametrize("m,k,n", PLACES)
@pytest.mark.parametrize("tiny", [1e-31, 1e-35, 1e-42])
def test_a_tiny_value_that_cannot_matter_sums_nothing_again(dev, m, k, n, tiny):
    """Values below 2^-100 among ordinary ones: the bits are those with zeros
    in their place (the f32 MFMA's sums differ in their rounding)."""
    from magnetar_hip import ops
    a, b = operands(m, k, n, m + 29)
    got = []
    for value in (0.0, tiny):
        a.reshape(-1)[:: 61] = value
        b[k // 2, 1::7] = value
        got.append(ops.matmul(dev, dev.upload(a), dev.upload(b)).numpy().view(np.uint32))
    assert np.array_equal(got[0], got[1])


@pytest.mark.parametrize("m,k,n", [(20, 480, 640), (31, 200, 258)])
@pytest.mark.parametrize("down", [-100, -108, -120])
@pytest.mark.parametrize("compact", [False, True])
def test_small_rows_of_a_panel_keep_their_precision(dev, m, k, n, down, compact):
    from magnetar_hip import ops
    a, b = operands(m, k, n, m + 31)
    a[::3] *= np.float32(2.0 ** down)
    b = (b * np.float32(2.0 ** 90)).view(np.uint32) & np.uint32(0xFFFF0000)
    half = (b >> 16).astype(np.uint16)
    b = b.view(np.float32)
    da = dev.upload(a)
    check(ops.matmul_bf16w(dev, da, dev.upload(half)).numpy() if compact else ops.matmul(dev, da, dev.upload(b)).numpy(), a, b)


@pytest.mark.parametrize("m,n", [(70, 70), (64, 2050), (2000, 2030), (4000, 4060), (20, 640), (9, 2), (31, 258)])
@pytest.mark.parametrize("compact", [False, True])
def test_one_and_two_products_keep_the_f32_error(dev, m, n, compact):
    """k 1 is a single rounded product, k 2 at most two products and a sum
    (an fma chain rounds less): bit for bit, and within 3 u of the terms."""
    from magnetar_hip import ops
    for k in (1, 2):
        a, b = operands(m, k, n, m + 37)
        if compact:
            b = (b.view(np.uint32) & np.uint32(0xFFFF0000)).view(np.float32)
        half = (b.view(np.uint32) >> 16).astype(np.uint16)
        da = dev.upload(a)
        got = ops.matmul_bf16w(dev, da, dev.upload(half)).numpy() if compact else ops.matmul(dev, da, dev.upload(b)).numpy()
        if k == 1:
            assert np.array_equal(got.view(np.uint32), (a * b).view(np.uint32))
        scale = np.abs(a).astype(np.float64) @ np.abs(b)
        assert np.all(np.abs(got - a.astype(np.float64) @ b.astype(np.float64)) <= k * 1.5 * 2.0 ** -24 * scale)


WORST = np.float32(1 + 2.0 ** -8 - 2.0 ** -17)  # its square's dropped products are 0.99 u of it


@pytest.mark.parametrize("m,k,n", [(70, 1, 70), (70, 3, 70), (2000, 16, 2030), (20, 3, 640), (4000, 72, 4060), (20, 480, 640),
                                   (300, 4096, 300)])
def test_operands_whose_dropped_products_are_largest(dev, m, k, n):
    """Every dropped product of the same sign and as large as any. Nothing but
    their sum and the rounding of the kept ones: (k / 16 * 6 + 2) u of the sum."""
    from magnetar_hip import ops
    a, b = np.full((m, k), WORST), np.full((k, n), WORST)
    got = ops.matmul(dev, dev.upload(a), dev.upload(b)).numpy()
    exact = k * np.float64(WORST) ** 2
    assert np.all(np.abs(got - exact) <= (k / 16 * 6 + 2) * 2.0 ** -24 * exact)

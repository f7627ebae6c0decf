"""Large fp32 products on the bf16 matrix cores (csrc/gemm_split.hip): every operand is the exact sum of
three bf16 numbers, elements that are not send their tile to the fp32 instruction."""
import numpy as np
import pytest

from conftest import capi

pytestmark = pytest.mark.gpu


def product(ctx, x, y, lay):
    """x [M, K] times y [N, K]^T; lay: "K" = stored with k contiguous, "R" = stored with the rows contiguous."""
    a = ctx.upload(x) if lay[0] == "K" else ctx.upload(np.ascontiguousarray(x.T)).transpose([1, 0])
    b = ctx.upload(y) if lay[1] == "K" else ctx.upload(np.ascontiguousarray(y.T)).transpose([1, 0])
    return a.replicate([y.shape[0]]).transpose([1, 0, 2]).contract(b.replicate([x.shape[0]]), 2)


def repeated(ctx, x, y, lay):
    """The values of `product`.  Small products are not formed from bf16 parts: as many of the same in a batch as make
    5e8 multiplications, all of which have to agree."""
    c = -(-500_000_000 // (x.size * y.shape[0]))
    stack = lambda v, how: (ctx.upload(np.stack([v] * c)) if how == "K" else ctx.upload(np.stack([np.ascontiguousarray(v.T)] * c)).transpose([0, 2, 1]))
    a, b = stack(x, lay[0]), stack(y, lay[1])
    out = a.replicate([y.shape[0]]).transpose([1, 2, 0, 3]).contract(b.replicate([x.shape[0]]).transpose([1, 0, 2, 3]), 3).numpy()
    assert np.array_equal(out, np.broadcast_to(out[:1], out.shape), equal_nan=True)
    return out[0]


def assert_close(out, x, y, k):
    """Sixteen products per rounded addition plus the roundings inside the sixteen and of the partial sums:
    at most (K / 16 + 16) half-ulps of the sum of magnitudes; the three terms left out stay under 2^-24 of it."""
    x, y = x.astype(np.float64), y.astype(np.float64)
    bound = (k / 16 + 17) * 2.0 ** -24 * (np.abs(x) @ np.abs(y).T) + 1e-45
    assert np.all(np.abs(out.astype(np.float64) - x @ y.T) <= bound)


@pytest.mark.parametrize("lay", ["KK", "KR", "RK", "RR"])
@pytest.mark.parametrize("m,n,k", [(128, 128, 1040), (129, 257, 1041), (300, 500, 1077), (255, 96, 2063), (2050, 514, 520), (97, 2300, 1025)])
def test_ragged_shapes(gpu, m, n, k, lay):
    rng = np.random.default_rng(m + n + k)
    x, y = rng.standard_normal((m, k)).astype(np.float32), rng.uniform(0, 1, (n, k)).astype(np.float32)
    gpu.profile(2)
    out = repeated(gpu, x, y, lay)
    labels = list(gpu.profile_report())
    gpu.profile(0)
    assert any(",split3,t128x128" in s for s in labels), labels
    assert_close(out, x, y, k)


@pytest.mark.parametrize("lay", ["KK", "KR", "RR"])
@pytest.mark.parametrize("k", [64, 65, 79, 80, 81, 95])
def test_few_steps(gpu, k, lay):
    """Loads run a step and splits half a step ahead: sums of a few steps, with and without a rest."""
    rng = np.random.default_rng(k)
    x, y = rng.standard_normal((130, k)).astype(np.float32), rng.standard_normal((100, k)).astype(np.float32)
    assert_close(repeated(gpu, x, y, lay), x, y, k)


@pytest.mark.parametrize("k", [20000, 20001, 20016, 20033, 20044])
def test_last_share_of_k(gpu, k):
    """K shared out: the last share is shorter than the others, down to less than a step."""
    rng = np.random.default_rng(k)
    x, y = rng.standard_normal((200, k)).astype(np.float32), rng.standard_normal((130, k)).astype(np.float32)
    gpu.profile(2)
    out = product(gpu, x, y, "KK").numpy()
    labels = list(gpu.profile_report())
    gpu.profile(0)
    assert any("split3" in s and ",s1," not in s for s in labels), labels
    assert_close(out, x, y, k)


@pytest.mark.parametrize("rest", [0.0, 2.0 ** -40])
@pytest.mark.parametrize("lay", ["KK", "RR"])
@pytest.mark.parametrize("diagonal", [False, True])
def test_rows_with_one_dominating_product(gpu, diagonal, lay, rest):
    """One rounding to fp32 and the three terms left out: 2 units of 2^-24 of the product.  The five small terms, at
    most 2^-7 of it, lose less than 2^-23 of themselves in each of five additions: 0.1 more with the tiny products."""
    m, n, k = 300, 280, 1040
    rng = np.random.default_rng(13)
    x, y = (rng.standard_normal((r, k)) * rest for r in (m, n))
    if diagonal:        # a matrix with a few large entries, one to a row, times an ordinary one
        x[np.arange(m), np.arange(m) * 3] = rng.uniform(1, 2, m)
        y = rng.standard_normal((n, k))
    else:
        x[:, 5], y[:, 5] = rng.uniform(1, 2, m), rng.uniform(1, 2, n)
    x, y = x.astype(np.float32), y.astype(np.float32)
    out, xd, yd = repeated(gpu, x, y, lay), x.astype(np.float64), y.astype(np.float64)
    mag = np.abs(xd) @ np.abs(yd).T
    top = np.abs(xd).max(1)[:, None] * np.abs(yd)[:, np.arange(m) * 3].T if diagonal else mag
    rows = top >= mag * (1 - 2.0 ** -20)     # (where the ordinary matrix holds something small the rest counts)
    assert np.count_nonzero(rows) > 0.95 * rows.size
    assert np.all(np.abs(out - xd @ yd.T)[rows] <= 2.1 * 2.0 ** -24 * mag[rows])


@pytest.mark.parametrize("scale", [1e-35, 1e-30, 1e30, 1.5e38])
def test_elements_that_three_bf16_cannot_hold(gpu, scale):
    """Tiny and huge operands: the products themselves stay in fp32's normal range."""
    m, n, k = 200, 300, 1030
    rng = np.random.default_rng(5)
    x = (rng.uniform(-1, 1, (m, k)) * scale).astype(np.float32)
    y = (rng.uniform(-1, 1, (n, k)) / scale / (64 if scale > 1 else 1)).astype(np.float32)
    out = repeated(gpu, x, y, "KR")
    xd, yd = x.astype(np.float64), y.astype(np.float64)
    # (the fp32 instruction rounds once per product)
    assert np.all(np.abs(out - xd @ yd.T) <= (k + 17) * 2.0 ** -24 * (np.abs(xd) @ np.abs(yd).T))


def test_infinities_and_nans_stay_where_they_belong(gpu):
    m, n, k = 260, 140, 1100
    rng = np.random.default_rng(6)
    x, y = rng.uniform(0.5, 1, (m, k)).astype(np.float32), rng.uniform(0.5, 1, (n, k)).astype(np.float32)
    x[3, 7], x[200, 1099], y[130, 0] = np.inf, np.nan, -np.inf
    out = repeated(gpu, x, y, "RK")
    want = x.astype(np.float64) @ y.astype(np.float64).T
    assert np.array_equal(np.isnan(out), np.isnan(want))
    assert np.array_equal(np.isposinf(out), np.isposinf(want)) and np.array_equal(np.isneginf(out), np.isneginf(want))
    fine = np.isfinite(want)
    assert np.all(np.abs(out[fine] - want[fine]) <= (k + 17) * 2.0 ** -24 * want[fine])


def test_products_close_to_the_largest_number(gpu):
    """Products that fit fp32 although the product of their operands' leading parts, both rounded up, does not."""
    m, n, k = 150, 200, 1030
    x, y = np.zeros((m, k), np.float32), np.zeros((n, k), np.float32)
    x[:, 1:], y[:, 1:] = 2.0 ** -40, 2.0 ** -41
    x[:, 0] = np.linspace(1.9961, 1.9999, m) * 2.0 ** 63
    y[:, 0] = np.linspace(1.9961, 1.9999, n) * 2.0 ** 63
    y[1::3, 0] *= -1
    out, want = repeated(gpu, x, y, "KK"), x.astype(np.float64) @ y.astype(np.float64).T
    assert np.all(np.abs(want) < 2.0 ** 128 * (1 - 2.0 ** -24)) and np.all(np.abs(want) > 2.0 ** 128 * (1 - 2.0 ** -8))
    assert np.all(np.abs(out - want) <= 4 * 2.0 ** -24 * np.abs(want))


@pytest.mark.parametrize("small", [2.0 ** -99, 2.0 ** -101, 2.0 ** -110, 2.0 ** -126, 2.0 ** -140, 2.0 ** -149])
def test_small_elements_keep_all_their_bits(gpu, small):
    """Down to the smallest subnormal number an element takes part with all the bits it has."""
    m, n, k = 140, 190, 1030
    rng = np.random.default_rng(11)
    x, y = (rng.uniform(1, 16, (m, k)) * small).astype(np.float32), rng.uniform(2.0 ** 20, 2.0 ** 21, (n, k)).astype(np.float32)
    x[::2, 1:] = 0
    out, xd, yd = repeated(gpu, x, y, "KR"), x.astype(np.float64), y.astype(np.float64)
    bound = np.where(np.arange(m) % 2 == 0, 4, k / 16 + 17)[:, None] * 2.0 ** -24 * (xd @ yd.T) + 2.0 ** -149
    assert np.all(np.abs(out - xd @ yd.T) <= bound)


@pytest.mark.parametrize("top_x,top_y", [(2.0 ** 103, 1.0), (2.0 ** 104, 1.0), (2.0 ** 60, 2.0 ** 10), (2.0 ** 40, 2.0 ** 40), (2.0 ** 62, 2.0 ** 62), (1.0, 2.0 ** 126)])
def test_large_elements_beside_ordinary_ones(gpu, top_x, top_y):
    """Either side of the limits from which a tile goes to the fp32 instruction."""
    m, n, k = 260, 150, 1040
    rng = np.random.default_rng(12)
    x, y = rng.uniform(-1, 1, (m, k)).astype(np.float32), rng.uniform(-1, 1, (n, k)).astype(np.float32)
    x[7, 3], x[200, 1039], y[140, 3] = top_x, -top_x * 0.7, top_y
    out, xd, yd = repeated(gpu, x, y, "RK"), x.astype(np.float64), y.astype(np.float64)
    # (the fp32 instruction rounds once per product)
    assert np.all(np.abs(out - xd @ yd.T) <= (k + 17) * 2.0 ** -24 * (np.abs(xd) @ np.abs(yd).T))


@pytest.mark.parametrize("terms", [2, 5])
def test_sum_of_products(gpu, terms):
    m, n, k = 130, 100, 2000
    rng = np.random.default_rng(terms)
    xs = [rng.standard_normal((m, k)).astype(np.float32) for _ in range(terms)]
    ys = [rng.standard_normal((n, k)).astype(np.float32) for _ in range(terms)]
    pairs = [(gpu.upload(x).replicate([n]).transpose([1, 0, 2]), gpu.upload(y).replicate([m])) for x, y in zip(xs, ys)]
    out = gpu.contract_sum(pairs, 2).numpy()
    assert_close(out, np.concatenate(xs, 1), np.concatenate(ys, 1), terms * k)


@pytest.mark.parametrize("batch,m,n,k,split", [(1, 128, 128, 1040, False), (3, 125, 194, 141, False), (1, 122, 113, 1251, False), (52, 101, 264, 107, True), (1, 441, 208, 3108, True)])
def test_small_products_are_left_to_the_fp32_instruction(gpu, batch, m, n, k, split):
    rng = np.random.default_rng(batch + k)
    x, y = rng.standard_normal((batch, m, k)).astype(np.float32), rng.standard_normal((batch, n, k)).astype(np.float32)
    gpu.profile(2)
    out = gpu.upload(x).replicate([n]).transpose([1, 2, 0, 3]).contract(gpu.upload(y).replicate([m]).transpose([1, 0, 2, 3]), 3).numpy()
    labels = list(gpu.profile_report())
    gpu.profile(0)
    assert any("split3" in s for s in labels) == split, labels
    xd, yd = x.astype(np.float64), y.astype(np.float64)
    # (the fp32 instruction rounds once per product)
    assert np.all(np.abs(out - xd @ yd.transpose(0, 2, 1)) <= (k + 17) * 2.0 ** -24 * (np.abs(xd) @ np.abs(yd).transpose(0, 2, 1)))

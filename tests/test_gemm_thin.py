"""fp32 products with 8 to 32 rows or columns under a long K: tiles of 128 x 32 on the bf16 matrix cores (csrc/gemm_split.hip)."""
import numpy as np
import pytest

import test_held_sums as held
from test_gemm_split import assert_close

pytestmark = pytest.mark.gpu


def operand(ctx, v, how, times, first):
    """v [rows, K] repeated along a kept dim: [rows, times, K] where it is the first factor, else [times, rows, K]."""
    a = ctx.upload(v) if how == "K" else ctx.upload(np.ascontiguousarray(v.T)).transpose([1, 0])
    a = a.replicate([times])
    return a.transpose([1, 0, 2]) if first else a


def sum_of(ctx, xs, ys, lay):
    m, n = xs[0].shape[0], ys[0].shape[0]
    ctx.profile(2)
    pairs = [(operand(ctx, x, lay[0], n, True), operand(ctx, y, lay[1], m, False)) for x, y in zip(xs, ys)]
    out = (ctx.contract_sum(pairs, 2) if len(pairs) > 1 else pairs[0][0].contract(pairs[0][1], 2)).numpy()
    labels = list(ctx.profile_report())
    ctx.profile(0)
    return out, any("t128x32" in s for s in labels), labels


@pytest.mark.parametrize("lay", ["KK", "KR", "RK", "RR"])
@pytest.mark.parametrize("m,n,k,terms", [
    (128, 32, 4096, 1),        # whole tiles
    (127, 31, 4099, 1),
    (129, 28, 1041, 5),        # a tile of one row
    (600, 8, 5003, 1),         # the fewest columns
    (9, 700, 4100, 1),         # the thin side first
    (33, 32, 129, 32),         # the fewest rows, a tail of one k
    (34, 30, 257, 20),         # shares of K with a tail
    (300, 17, 20000, 2),       # long shares: four blocks for a CU
    (256, 32, 65536, 1),       # the longest K
])
def test_ragged_shapes(gpu, m, n, k, terms, lay):
    rng = np.random.default_rng(m + n + k)
    xs = [rng.standard_normal((m, k)).astype(np.float32) for _ in range(terms)]
    ys = [rng.uniform(0, 1, (n, k)).astype(np.float32) for _ in range(terms)]
    out, taken, labels = sum_of(gpu, xs, ys, lay)
    assert taken, labels
    assert_close(out, np.concatenate(xs, 1), np.concatenate(ys, 1), terms * k)


@pytest.mark.parametrize("m,n,k,terms", [(700, 7, 4096, 1), (300, 33, 4096, 1), (32, 32, 500, 20), (300, 32, 4095, 1), (300, 20, 65537, 1)])
def test_what_other_kernels_keep(gpu, m, n, k, terms):
    rng = np.random.default_rng(k)
    xs, ys = ([rng.standard_normal((r, k)).astype(np.float32) for _ in range(terms)] for r in (m, n))
    out, taken, labels = sum_of(gpu, xs, ys, "KK")
    assert not taken, labels
    x, y = (np.concatenate(v, 1).astype(np.float64) for v in (xs, ys))
    # (the fp32 instruction rounds once per product)
    assert np.all(np.abs(out - x @ y.T) <= (terms * k + 17) * 2.0 ** -24 * (np.abs(x) @ np.abs(y).T))


def test_infinities_nans_and_large_elements(gpu):
    """Tiles that meet them are formed by the fp32 instruction; the others are not touched."""
    m, n, k = 300, 29, 4111
    rng = np.random.default_rng(2)
    x, y = rng.uniform(0.5, 1, (m, k)).astype(np.float32), rng.uniform(0.5, 1, (n, k)).astype(np.float32)
    x[3, 7], x[140, 4110], x[280, 0], y[28, 2000] = np.inf, np.nan, 2.0 ** 110, -2.0 ** 100
    out, taken, labels = sum_of(gpu, [x], [y], "KR")
    assert taken, labels
    with np.errstate(invalid="ignore"):
        xd, yd = x.astype(np.float64), y.astype(np.float64)
        want, mag = xd @ yd.T, np.abs(xd) @ np.abs(yd).T
        want = np.where(np.abs(want) >= 2.0 ** 128, np.sign(want) * np.inf, want)
    assert np.array_equal(np.isnan(out), np.isnan(want))
    assert np.array_equal(np.isposinf(out), np.isposinf(want)) and np.array_equal(np.isneginf(out), np.isneginf(want))
    fine = np.isfinite(want)
    assert np.all(np.abs(out[fine] - want[fine]) <= (k + 17) * 2.0 ** -24 * mag[fine])


@pytest.mark.parametrize("lay", ["KK", "RK"])
def test_products_of_a_recording(lay):
    held.test_products_of_a_recording_go_out_together(held.pkg.hostapi.Host(), np.float32, [(130, 28, 5000), (130, 32, 5000), (128, 128, 30000), (500, 17, 9001)], lay)


@pytest.mark.parametrize("lay", ["KK", "RR"])
@pytest.mark.parametrize("m,n,k", [(300, 28, 4100), (9, 700, 4100)])
def test_one_dominating_product(gpu, m, n, k, lay):
    """A sum that is one product is that product rounded: the parts of both factors are multiplied with one another but for the last with
    the last (2^-34 of the product), and the small ones, 2^-7 of it, lose less than 2^-23 of themselves in each of seven additions."""
    rng = np.random.default_rng(m)
    x, y = np.zeros((m, k), np.float32), np.zeros((n, k), np.float32)
    x[:, 7], y[:, 7] = rng.uniform(1, 2, m), rng.uniform(1, 2, n)
    out, taken, labels = sum_of(gpu, [x], [y], lay)
    assert taken, labels
    want = x.astype(np.float64) @ y.astype(np.float64).T
    assert np.max(np.abs(out - want) / want) <= (1 + 7 * 2.0 ** -6 + 2.0 ** -9) * 2.0 ** -24

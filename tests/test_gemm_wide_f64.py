"""fp64 products addressed by one stride per index (csrc/gemm_wide_f64.hip)."""
import numpy as np
import pytest

from test_gemm_split import product

pytestmark = pytest.mark.gpu


def assert_close(out, x, y, k):
    """Against numpy's fp64 product: each side rounds once per product and per addition at most."""
    bound = 2 * (k + 8) * 2.0 ** -53 * (np.abs(x) @ np.abs(y).T)
    assert np.all(np.abs(out - x @ y.T) <= bound)


@pytest.mark.parametrize("lay", ["KK", "KR", "RK", "RR"])
@pytest.mark.parametrize("m,n,k", [(128, 64, 1040), (64, 64, 1025), (65, 129, 1041), (300, 500, 1077), (127, 191, 2063), (1000, 1025, 513), (2050, 514, 520),
                                   (97, 4300, 1151), (2048, 2050, 64), (4097, 1000, 77)])
def test_ragged_shapes(gpu, m, n, k, lay):
    """Tiles with one row, chunks of K that end anywhere within a step, an odd and an even number of steps."""
    rng = np.random.default_rng(m + n + k)
    x, y = rng.standard_normal((m, k)), rng.uniform(0, 1, (n, k))
    gpu.check(gpu.lib.profile_enable(gpu.h, 2))
    out = product(gpu, x, y, lay).numpy()
    labels = list(gpu.profile_report())
    gpu.check(gpu.lib.profile_enable(gpu.h, 0))
    assert any(",wide," in s for s in labels), labels
    assert_close(out, x, y, k)


@pytest.mark.parametrize("k", [1089, 1100, 1104, 1120, 1121])
def test_every_way_a_chunk_can_end(gpu, k):
    rng = np.random.default_rng(k)
    x, y = rng.standard_normal((2100, k)), rng.standard_normal((700, k))
    assert_close(product(gpu, x, y, "KR").numpy(), x, y, k)


def test_infinities_and_nans_stay_where_they_belong(gpu):
    m, n, k = 260, 140, 1100
    rng = np.random.default_rng(6)
    x, y = rng.uniform(0.5, 1, (m, k)), rng.uniform(0.5, 1, (n, k))
    x[3, 7], x[200, 1099], x[259, 0], y[130, 0] = np.inf, np.nan, 1e308, -np.inf
    for lay in ("RK", "KR"):
        out, want = product(gpu, x, y, lay).numpy(), x @ y.T
        assert np.array_equal(np.isnan(out), np.isnan(want))
        assert np.array_equal(np.isposinf(out), np.isposinf(want)) and np.array_equal(np.isneginf(out), np.isneginf(want))
        fine = np.isfinite(want)
        assert np.all(np.abs(out[fine] - want[fine]) <= 2 * (k + 8) * 2.0 ** -53 * np.abs(want[fine]))


@pytest.mark.parametrize("terms", [2, 5])
def test_sums_and_batches_of_products(gpu, terms):
    rng = np.random.default_rng(terms)
    m, n, k = 150, 130, 1037
    x, y = rng.standard_normal((terms, m, k)), rng.standard_normal((terms, n, k))
    a, b = gpu.upload(x), gpu.upload(y)
    pairs = [(a.index_prefix([t]).replicate([n]).transpose([1, 0, 2]), b.index_prefix([t]).replicate([m])) for t in range(terms)]
    got = gpu.contract_sum(pairs, 2).numpy()
    bound = 2 * (terms * k + 8) * 2.0 ** -53 * np.einsum("tmk,tnk->mn", np.abs(x), np.abs(y))
    assert np.all(np.abs(got - np.einsum("tmk,tnk->mn", x, y)) <= bound)
    batch = a.replicate([n]).transpose([1, 2, 0, 3]).contract(b.replicate([m]).transpose([1, 0, 2, 3]), 3).numpy()
    for t in range(terms):
        assert_close(batch[t], x[t], y[t], k)

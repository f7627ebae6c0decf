"""Sums along rows that lie side by side in memory, 16 bytes a load (csrc/contract.hip, wide_sum)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dt", [np.float64, np.float32])
@pytest.mark.parametrize("rows,n", [(1, 1), (3, 63), (5, 255), (2, 257), (70, 1023), (9, 1025), (300, 4099), (2100, 1031), (1025, 1024), (4095, 1500), (130, 70001), (1, 1000003)])
def test_rows_that_start_anywhere(gpu, dt, rows, n):
    """Whole tables, tables without their first or last columns (rows off 16-byte boundaries), reversed rows (the other path); plain
    sums, products with another table, with ones that are one element, and with one row for all."""
    rng = np.random.default_rng(n)
    x, y = (rng.uniform(-1, 1, (rows, n + 3)).astype(dt) for _ in range(2))
    a, b = gpu.upload(x), gpu.upload(y)
    two = gpu.upload(np.asarray(2.0, dt)).replicate([rows, n])
    for lo in (0, 1, 3):
        av, bv, xv, yv = a.slice(1, lo, n), b.slice(1, 3 - lo, n), x[:, lo:lo + n].astype(np.float64), y[:, 3 - lo:3 - lo + n].astype(np.float64)
        row = b.index_prefix([0]).slice(0, lo, n).replicate([rows])
        yrow = y[0, lo:lo + n].astype(np.float64)
        for got, terms in ((av.contract(None, 1), xv), (av.contract(bv, 1), xv * yv), (av.contract(two, 1), 2 * xv), (av.contract(row, 1), xv * yrow),
                           (av.reverse(1).contract(bv, 1), xv[:, ::-1] * yv), (av.contract(bv, 0), (xv * yv).reshape(1, -1))):
            want, mag = terms.sum(-1), np.abs(terms).sum(-1)
            # summed in fp64 either way (a rounding per product and per addition), rounded once to the result's type
            m = terms.shape[-1]
            assert np.all(np.abs(got.numpy().reshape(want.shape) - want) <= 2 * (m + 4) * 2.0 ** -53 * mag + np.finfo(dt).eps * np.abs(want))


def test_infinities_times_one_element(gpu):
    x = np.ones((3, 5000))
    x[0, 7], x[1, 4999], x[2, 100], x[2, 200] = np.inf, np.nan, np.inf, -np.inf
    a = gpu.upload(x)
    ones = gpu.upload(np.asarray(1.0)).replicate([3, 5000])
    zeros = gpu.upload(np.asarray(0.0)).replicate([3, 5000])
    assert np.array_equal(a.contract(ones, 1).numpy(), [np.inf, np.nan, np.nan], equal_nan=True)
    assert np.all(np.isnan(a.contract(zeros, 1).numpy()))

"""A few rows of some hundred to some thousand elements (csrc/contract.hip): extrema by a block per row, sums of many
partial sums by a block per output."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dt", [np.float64, np.float32, np.int64, np.int8])
@pytest.mark.parametrize("rows,n", [(1, 511), (1, 512), (1, 513), (3, 1024), (64, 1025), (65, 1025), (2, 8191), (1, 9217)])
def test_first_extremum(gpu, dt, rows, n):
    """Ties: the first position wins, within a lane's own positions and between lanes; rows contiguous and strided."""
    rng = np.random.default_rng(n)
    x = rng.integers(-100 if dt == np.int8 else -n, 100 if dt == np.int8 else n, (rows, n)).astype(dt)
    x[0, n // 3] = x[0, -1] = x[0].max()
    x[-1, 5] = x[-1, n // 2] = x[-1].min()
    for a in (gpu.upload(x), gpu.upload(np.ascontiguousarray(x.T)).transpose([1, 0])):
        for want_max in (True, False):
            vals, idx = a.extremum_last(want_max)
            want = (np.argmax if want_max else np.argmin)(x, axis=-1)
            assert np.array_equal(idx.numpy(), want)
            assert np.array_equal(vals.numpy(), np.take_along_axis(x, want[:, None], 1)[:, 0])


def test_extrema_beside_nans(gpu):
    """Element after element with > or <, as the checker goes: a NaN is passed over, and stays when it is the first."""
    x = np.random.default_rng(4).uniform(-1, 1, (5, 1500))
    x[0, 1:1400:2] = np.nan
    x[1, 0] = np.nan
    x[2, 1:] = np.nan
    x[3, 1023], x[3, 70] = np.nan, np.inf
    x[4, 1:1025] = np.nan
    for want_max in (True, False):
        vals, idx = gpu.upload(x).extremum_last(want_max)
        want = (np.nanargmax if want_max else np.nanargmin)(x, axis=-1)
        want[1] = 0
        assert np.array_equal(idx.numpy(), want)
        assert np.array_equal(vals.numpy(), np.take_along_axis(x, want[:, None], 1)[:, 0], equal_nan=True)


@pytest.mark.parametrize("dt", [np.float64, np.float32, np.int64])
@pytest.mark.parametrize("outs,n", [(1, 3000001), (7, 600000), (300, 40000)])
def test_sums_of_many_partial_sums(gpu, dt, outs, n):
    rng = np.random.default_rng(outs)
    x = (rng.integers(-9, 9, (outs, n)) if dt == np.int64 else rng.uniform(-1, 1, (outs, n))).astype(dt)
    got = gpu.upload(x).contract(None, 1).numpy()
    wide = x.astype(np.int64 if dt == np.int64 else np.float64)
    if dt == np.int64:
        assert np.array_equal(got, wide.sum(1))
    else:      # summed in fp64 by either, rounded once to the result's type
        assert np.all(np.abs(got - wide.sum(1)) <= n * 2.0 ** -52 * np.abs(wide).sum(1) / 100 + np.finfo(dt).eps * np.abs(wide.sum(1)))


@pytest.mark.parametrize("dt", [np.float64, np.float32, np.int64, np.int8])
def test_rows_of_the_types_own_extremum(gpu, dt):
    """Nothing exceeds it: the first place, and the first one that does where there is one."""
    lo, hi = (-np.inf, np.inf) if np.dtype(dt).kind == "f" else (np.iinfo(dt).min, np.iinfo(dt).max)
    for want_max, end in ((True, lo), (False, hi)):
        x = np.full((4, 1500), end, dt)
        x[1, 1499] = x[2, 1030] = x[2, 1200] = 3
        if np.dtype(dt).kind == "f":
            x[3, 1:] = np.nan
            x[0, 5::2] = np.nan
        vals, idx = gpu.upload(x).extremum_last(want_max)
        assert idx.numpy().tolist() == [0, 1499, 1030, 0]
        assert np.array_equal(vals.numpy(), np.array([end, 3, 3, end], dt))


@pytest.mark.parametrize("dt", [np.float64, np.float32])
@pytest.mark.parametrize("rows,n", [(1, 16383), (1, 16384), (3, 50001), (16, 131073), (3, 300), (70, 700)])
def test_extrema_beside_nans_whoever_shares_a_row(gpu, dt, rows, n):
    """One rule for a block, for pieces of a row and for a wavefront: a NaN that comes first in a row stays, any other is no candidate --
    first of a piece, first of a lane, or of every lane; nothing but NaNs behind the first element."""
    rng = np.random.default_rng(n)
    base = rng.uniform(-1, 1, (rows, n)).astype(dt)
    pieces = max(1, min(128, n // 1024))
    step = (n + pieces - 1) // pieces
    hidden = min(n - 1, 64 if n < 1024 else 256)      # of the lane that met the NaN first
    cases = []
    x = base.copy()
    x[-1, 0] = np.nan
    cases.append(x)
    for end in (5, -5):
        x = base.copy()
        x[:, step::step] = np.nan
        x[:, (step if n > step else 0) + hidden - (0 if n > step else 1)] = end
        cases.append(x)
        x = base.copy()
        x[:, 1:hidden + 1] = np.nan
        x[:, min(n - 1, 2 * hidden)] = end
        cases.append(x)
    x = base.copy()
    x[0, 1:] = np.nan
    cases.append(x)
    cases.append(np.full((rows, n), np.nan, dt))
    for x in cases:
        seen = np.where(np.isnan(x[:, :1]), np.arange(n) == 0, ~np.isnan(x))
        for want_max in (True, False):
            vals, idx = gpu.upload(x).extremum_last(want_max)
            want = np.where(seen, np.nan_to_num(x) if want_max else -np.nan_to_num(x), -np.inf).argmax(1)
            assert np.array_equal(idx.numpy(), want)
            assert np.array_equal(vals.numpy(), np.take_along_axis(x, want[:, None], 1)[:, 0], equal_nan=True)

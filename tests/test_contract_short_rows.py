"""Reductions over several dims, and ones whose results lie along memory (lane_body, flat_sum and rows_sum, csrc/contract.hip), at the
edges of a block's 256 results, of the 256 indices whose offsets are kept, of the loads that go together, and of a wavefront's 64 lanes."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def data(rng, shape, dt):
    if np.issubdtype(dt, np.integer):
        return rng.integers(-50, 50, shape).astype(dt)
    return rng.uniform(-1, 1, shape).astype(dt)


def compare(got, x, y, axes, dt):
    p = x if y is None else x * y if np.issubdtype(dt, np.integer) else x.astype(np.longdouble) * y
    if np.issubdtype(dt, np.integer):
        assert np.array_equal(got, p.sum(axes, dtype=dt))
        return
    p = p.astype(np.longdouble)
    n = np.prod([p.shape[k] for k in axes])
    # every sum of n products in 64 bits, in any order, then one rounding to the result's type
    bound = n * 2.0 ** -53 * np.abs(p).sum(axes) + np.finfo(dt).eps * np.abs(p.sum(axes))
    assert np.all(np.abs(got - p.sum(axes)) <= bound)


@pytest.mark.parametrize("n_out", [2048, 2049, 2303, 5000])
@pytest.mark.parametrize("R", [(1,), (7,), (3, 3), (17, 15), (16, 16), (257,), (5, 120), (3, 2, 200)])
@pytest.mark.parametrize("dt", [np.float64, np.float32, np.int32])
def test_results_along_memory(gpu, n_out, R, dt):
    rng = np.random.default_rng(n_out)
    shape = R + (n_out,)
    x, y = data(rng, shape, dt), data(rng, shape, dt)
    axes = tuple(range(len(R)))
    perm = [len(R)] + list(axes)
    a, b = gpu.upload(x), gpu.upload(y)
    compare(a.transpose(perm).contract(None, 1).numpy(), x, None, axes, dt)
    compare(a.transpose(perm).contract(b.transpose(perm), 1).numpy(), x, y, axes, dt)
    if len(R) == 2:            # the second operand's dims in another order
        z = data(rng, (R[1], R[0], n_out), dt)
        compare(a.transpose(perm).contract(gpu.upload(z).transpose([2, 1, 0]), 1).numpy(), x, z.transpose(1, 0, 2), axes, dt)


@pytest.mark.parametrize("terms", [2, 5])
def test_several_terms_along_memory(gpu, terms):
    rng = np.random.default_rng(terms)
    x, y = rng.uniform(-1, 1, (2, terms, 9, 37, 2100))
    pairs = [(gpu.upload(x[t]).transpose([2, 0, 1]), gpu.upload(y[t]).transpose([2, 0, 1])) for t in range(terms)]
    got = gpu.contract_sum(pairs, 1).numpy()
    compare(got, x, y, (0, 1, 2), np.float64)


@pytest.mark.parametrize("n_out,Q", [(64, 700), (300, 41), (300, 3), (2000, 2), (2000, 5), (5, 1300), (1, 9)])
@pytest.mark.parametrize("Lin", [2, 5, 63, 64, 65, 300])
@pytest.mark.parametrize("dt", [np.float64, np.float32, np.int64])
def test_short_rows(gpu, n_out, Q, Lin, dt):
    rng = np.random.default_rng(Q)
    x, y = data(rng, (Q, n_out, Lin), dt), data(rng, (Q, n_out, Lin), dt)
    a, b = gpu.upload(x).transpose([1, 0, 2]), gpu.upload(y).transpose([1, 0, 2])
    compare(a.contract(None, 1).numpy(), x, None, (0, 2), dt)
    compare(a.contract(b, 1).numpy(), x, y, (0, 2), dt)


def test_short_rows_of_infinities(gpu):
    """A lane without an element adds nothing: its place in the last round reads another's, which may not be a number."""
    x = np.zeros((7, 300, 30))
    x[0, 5, 0], x[3, 9, 29], x[6, 20, 29] = np.inf, -np.inf, np.nan
    got = gpu.upload(x).transpose([1, 0, 2]).contract(None, 1).numpy()
    want = x.sum((0, 2))
    assert np.array_equal(got, want, equal_nan=True)

"""Row sums in double precision from a waiting product's blocks (csrc/gemm_wide_f64.hip), and sums of the rows of several terms by one
launch (k_row_terms in csrc/contract.hip): against long doubles, within n 2^-53 of the sum of magnitudes and a rounding of the type."""
import numpy as np
import pytest

import test_held_sums as held

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def host():
    return held.pkg.hostapi.Host()


def summed(one, xs):
    s = xs[0].sdot1In(one)
    for x in xs[1:]:
        s = s + x.sdot1In(one)
    return s


@pytest.mark.parametrize("lay", ["K", "R"])
@pytest.mark.parametrize("first", ["products", "sums"])
@pytest.mark.parametrize("terms,m,n,k", [(2, 64, 64, 10000), (3, 65, 130, 3001), (28, 128, 128, 150), (2, 300, 784, 2500), (5, 128, 64, 79), (2, 100, 300, 1101)])
@pytest.mark.parametrize("f", [1.0, np.inf, -0.75])
def test_rows_with_a_product(host, terms, m, n, k, first, lay, f):
    """Every element times the factor, none of the zeros behind the end of K (an infinite factor shows them).  A sum asked for
    before the product is a launch of its own, and so is one of a single term."""
    rng = np.random.default_rng(m + n)
    xs = [rng.uniform(0.5, 1, (m, k)) * rng.choice([-1, 1], (m, 1)) for _ in range(terms)]
    ys = [rng.uniform(0, 1, (k, n) if lay == "R" else (n, k)) for _ in range(terms)]
    xs[-1][3, k - 1], xs[0][7, 0], xs[0][9, 5], xs[0][9, 6], xs[1][11, 2] = np.inf, np.nan, np.inf, -np.inf, 0.0
    a, b = [host.concrete(x) for x in xs], [host.concrete(y) if lay == "R" else host.concrete(y).stranspose([1, 0]) for y in ys]
    one = host.concrete(np.asarray(f)).sreplicate(k).sreplicate(m)

    def program():
        p = a[0].smatmul2(b[0])
        for u, v in zip(a[1:], b[1:]):
            p = p + u.smatmul2(v)
        if first == "products":
            held.force(host, p)
        return [summed(one, a[::-1]), a[0].sdot1In(one), p]

    with np.errstate(invalid="ignore"):
        v = np.stack(xs).astype(np.longdouble) * f
        want = [v.sum((0, 2)).astype(np.float64), v[0].sum(1).astype(np.float64)]
        size = [np.abs(v).sum((0, 2)).astype(np.float64), np.abs(v[0]).sum(1).astype(np.float64)]
    eager = [v.numpy() for v in program()]
    graph, res, labels = held.recorded(host, program)
    assert sum(q.count("+rows") * c for q, c in labels.items()) == (first == "products"), labels
    try:
        for _ in range(3):
            graph.launch()
            got = [v.numpy() for v in res]
            assert np.array_equal(got[2], eager[2], equal_nan=True)
            for g, w, s in zip(got, want, size):
                fine = np.isfinite(w)
                assert np.array_equal(g[~fine], w[~fine], equal_nan=True)
                assert np.all(np.abs(g[fine] - w[fine]) <= 2 * (terms * k + 8) * 2.0 ** -53 * s[fine])
            [v.numpy() for v in program()]
    finally:
        graph.free()


@pytest.mark.parametrize("dt", [np.float64, np.float32])
@pytest.mark.parametrize("terms,m,k,launches", [(2, 16, 1, 0), (2, 16, 2, 1), (3, 15, 40, 0), (5, 33, 63, 1), (28, 128, 150, 1), (32, 17, 129, 1), (32, 40, 512, 1), (32, 40, 513, 0), (33, 40, 128, 1), (9, 64, 257, 1)])
def test_rows_of_terms(gpu, dt, terms, m, k, launches):
    """Around the launch's limits: 16 rows, 16384 elements to a row; terms with rows further apart than they are long; a factor."""
    rng = np.random.default_rng(terms * m)
    xs = [rng.uniform(-1, 1, (m, k + 3)).astype(dt) for _ in range(terms)]
    xs[-1][2, 1 % k] = np.inf
    for f in (1.0, -0.7):
        one = gpu.upload(np.asarray(f, dt)).replicate([m, k])
        for lo in (0, 3):
            pairs = [(gpu.upload(x).slice(1, lo, k), one) for x in xs]
            gpu.profile(True)
            s = gpu.contract_sum(pairs, 1)
            got = s.numpy()
            n = gpu.profile_report().get("row_terms", (0,))[0]
            gpu.profile(False)
            assert n == launches, n
            cut = np.stack([x[:, lo:lo + k] for x in xs]).astype(np.float64)
            v = cut * float(dt(f))
            with np.errstate(invalid="ignore"):
                want, size = v.sum((0, 2)), np.abs(v).sum((0, 2))
            fine = np.isfinite(want)
            assert np.array_equal(got[~fine], want[~fine].astype(dt), equal_nan=True)
            bound = (np.finfo(dt).eps * (1 + terms // 32) + 2 * (terms * k + 8) * 2.0 ** -53) * size
            assert got.dtype == dt and np.all(np.abs(got[fine] - want[fine]) <= bound[fine])

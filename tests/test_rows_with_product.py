"""Sums of the rows that a waiting fp32 product multiplies come from that product's blocks (csrc/gemm_split.hip) in a recording."""
import ctypes as C
import threading

import numpy as np
import pytest

import test_held_sums as held

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def host():
    return held.pkg.hostapi.Host()


def check(host, program, want, size, n, joined):
    """`joined` of the recording's sums come from a product's blocks.  Every replay against what the program gives submitted one by one, where row sums are launches of their own: both are sums in
    doubles, rounded once to fp32, and once more for each of at most two additions of results."""
    eager = [v.numpy() for v in program()]
    graph, res, labels = held.recorded(host, program)
    assert sum(k.count("+rows") * v for k, v in labels.items()) == joined, labels
    bound = [4 * (2.0 ** -24 + n * 2.0 ** -53) * s for s in size]
    try:
        for _ in range(3):
            graph.launch()
            host.sync()
            for got, e in list(zip(res, eager))[len(want):]:      # the products themselves: bit for bit
                assert np.array_equal(got.numpy(), e, equal_nan=True)
            for got, e, w, b in zip(res, eager, want, bound):
                got = got.numpy()
                fine = np.isfinite(w)
                assert np.array_equal(got[~fine], w[~fine].astype(np.float32), equal_nan=True)
                assert np.all(np.abs(got[fine] - w[fine]) <= b[fine]) and np.all(np.abs(got[fine] - e[fine]) <= b[fine])
            [v.numpy() for v in program()]
    finally:
        graph.free()


def rows(a):
    return a.stranspose([1, 0]).ssum()


@pytest.mark.parametrize("lay", ["K", "R"])
@pytest.mark.parametrize("first", ["products", "sums"])
@pytest.mark.parametrize("m,n,k", [(128, 128, 30000), (129, 300, 20011), (300, 784, 5000), (2050, 130, 4099), (128, 28, 35000), (257, 9, 20003), (34, 32, 9001)])
def test_row_sums(host, m, n, k, first, lay):
    """Whole and ragged tiles of both widths, several columns of tiles, a tail of K; two sums of the same rows, of other rows and of
    rows of which a part is multiplied; rows with infinities and NaNs.  A sum that is asked for before the products are is a launch of its own."""
    rng = np.random.default_rng(m)
    x, z = (rng.uniform(-1, 1, (m, k)).astype(np.float32) for _ in range(2))
    y = rng.uniform(0, 1, (k, n) if lay == "R" else (n, k)).astype(np.float32)
    x[3, k - 1], x[7, 0], x[9, 5], x[9, 6] = np.inf, np.nan, np.inf, -np.inf
    z[5, 11] = -np.inf
    a, c, b = host.concrete(x), host.concrete(z), host.concrete(y)
    if lay == "K":
        b = b.stranspose([1, 0])

    def program():
        products = [a.smatmul2(b), c.smatmul2(b)]
        if first == "products":
            held.force(host, *products)
        return [rows(a), rows(c), rows(a) + rows(c), -rows(a)] + products

    with np.errstate(invalid="ignore"):
        sx, sz = x.astype(np.float64).sum(1), z.astype(np.float64).sum(1)
        want = [sx, sz, sx + sz, -sx]
        size = [np.abs(x).sum(1, dtype=np.float64), np.abs(z).sum(1, dtype=np.float64)]
    size += [size[0] + size[1], size[0]]

    check(host, program, want, size, k, 2 if first == "products" else 0)


def test_operand_written_between(host):
    """Rows that are overwritten after the product was submitted: the sum is that of what they hold when it is asked for."""
    rng = np.random.default_rng(1)
    m, n, k = 128, 128, 20000
    x, y, z = (rng.uniform(-1, 1, s).astype(np.float32) for s in ((m, k), (k, n), (m, k)))
    a, b, c = (host.concrete(v) for v in (x, y, z))

    def program():
        a.assign(c)
        p = a.smatmul2(b)
        held.force(host, p)
        s = rows(a)
        return [p, s]

    [v.numpy() for v in program()]
    graph, (p, s), labels = held.recorded(host, program)
    assert any("+rows" in k for k in labels), labels
    try:
        for _ in range(3):
            a.overwrite(x)
            graph.launch()
            host.sync()
            w = z.astype(np.float64)
            assert np.all(np.abs(s.numpy() - w.sum(1)) <= 4 * (2.0 ** -24 + k * 2.0 ** -53) * np.abs(w).sum(1))
            assert np.all(np.abs(p.numpy() - w @ y) <= (k / 16 + 17) * 2.0 ** -24 * (np.abs(w) @ np.abs(y.astype(np.float64))))
    finally:
        graph.free()


def test_sums_of_terms(host):
    """A recurrence's weight and bias gradients: several products into one, and the sum of all their rows."""
    rng = np.random.default_rng(2)
    m, n, k, t = 130, 96, 5000, 6
    xs, ys = [rng.uniform(-1, 1, (m, k)).astype(np.float32) for _ in range(t)], [rng.uniform(-1, 1, (k, n)).astype(np.float32) for _ in range(t)]
    a, b, one = [host.concrete(x) for x in xs], [host.concrete(y) for y in ys], host.concrete(np.ones((), np.float32))

    def program():
        p = a[0].smatmul2(b[0])
        for u, v in zip(a[1:], b[1:]):
            p = p + u.smatmul2(v)
        held.force(host, p)
        ones = one.sreplicate(k).sreplicate(m)
        s = a[-1].sdot1In(ones)
        for u in a[-2::-1]:      # (in the other order)
            s = s + u.sdot1In(ones)
        return [s, p.ssum()]

    x64 = np.concatenate(xs, 1).astype(np.float64)
    w, mag = x64.sum(1), np.abs(x64).sum(1)
    eager = [v.numpy() for v in program()]
    graph, (s, q), labels = held.recorded(host, program)
    assert any("+rows" in k for k in labels), labels
    try:
        for _ in range(3):
            graph.launch()
            host.sync()
            assert np.all(np.abs(s.numpy() - w) <= 4 * ((t + 1) * 2.0 ** -24 + t * k * 2.0 ** -53) * mag)
            assert np.array_equal(q.numpy(), eager[1])
    finally:
        graph.free()


@pytest.mark.parametrize("m,n,k", [(128, 128, 30000), (129, 28, 20011)])
@pytest.mark.parametrize("f", [np.inf, -0.75, 0.0, 3e38])
def test_factor_of_a_row_sum(host, m, n, k, f):
    """Every element is multiplied before it is added: an infinite factor over a row that has a zero, or both signs, gives no number."""
    rng = np.random.default_rng(m)
    x, y = rng.uniform(0.5, 1, (m, k)).astype(np.float32), rng.uniform(0, 1, (k, n)).astype(np.float32)
    x[1, 17], x[2, k - 1], x[5, :2], x[m - 1, 0] = 0.0, -1.0, (np.inf, -np.inf), np.nan
    a, b, c = host.concrete(x), host.concrete(y), host.concrete(np.asarray(f, np.float32))

    def program():
        p = a.smatmul2(b)
        held.force(host, p)
        return [a.sdot1In(c.sreplicate(k).sreplicate(m)), p]

    with np.errstate(invalid="ignore"):
        terms = x.astype(np.float64) * np.float64(np.float32(f))
        want, size = terms.sum(1), np.abs(terms).sum(1)
        big = np.where(np.abs(want) >= 2.0 ** 128, np.sign(want) * np.inf, want)
    check(host, program, [big], [size], k, 1)


@pytest.mark.parametrize("dt,terms,m,n,k", [(np.float32, 1, 128, 128, 30000), (np.float32, 6, 130, 96, 5000), (np.float64, 3, 65, 130, 3001)])
@pytest.mark.parametrize("by", ["gather", "extremum"])
def test_factor_that_waits(host, dt, terms, m, n, k, by):
    """The factor is the result of a launch that is held back by itself: it goes out before the product that reads it, also where
    something sends that product out which does not read the factor."""
    rng = np.random.default_rng(m)
    xs, ys = [rng.uniform(0.5, 1, (m, k)).astype(dt) for _ in range(terms)], [rng.uniform(0, 1, (k, n)).astype(dt) for _ in range(terms)]
    a, b = [host.concrete(x) for x in xs], [host.concrete(y) for y in ys]
    values = rng.uniform(1, 2, 100).astype(dt)
    table, at = host.concrete(values), host.concrete(np.asarray(3, np.int64))

    def program():
        p = a[0].smatmul2(b[0])
        for u, v in zip(a[1:], b[1:]):
            p = p + u.smatmul2(v)
        held.force(host, p)
        f = table.sgather((), lambda: [at.lift(())]) if by == "gather" else held.pkg.workloads.sminimum(table)
        held.force(host, f)
        by_f = f.sreplicate(k).sreplicate(m)
        s = a[0].sdot1In(by_f)
        for u in a[1:]:
            s = s + u.sdot1In(by_f)
        held.force(host, s)
        q = p * 2.0
        held.force(host, q)
        return [s, q]

    total, size = sum(x.sum(1, dtype=np.longdouble) for x in xs).astype(np.float64), 2.0 * sum(np.abs(x).sum(1, dtype=np.float64) for x in xs)
    [v.numpy() for v in program()]
    graph, (s, q), labels = held.recorded(host, program)
    assert any("+rows" in v for v in labels), labels
    try:
        for i in (5, 70, 11, 70):
            at.overwrite(np.asarray(i, np.int64))
            now = values.copy()
            now[20] = i / 128
            table.overwrite(now)
            f = float(now[i] if by == "gather" else now.min())
            graph.launch()
            host.sync()
            assert np.all(np.abs(s.numpy() - f * total) <= 2 * (2.0 ** (-24 if dt == np.float32 else -53) + terms * k * 2.0 ** -53) * size), i
            [v.numpy() for v in program()]
    finally:
        graph.free()


def test_two_threads_ask_for_the_same_rows():
    """One of the sums joins the product, the other is a launch of its own."""
    ctx = held.pkg.capi.Lib().context(0)
    m, n, k = 256, 64, 20000
    rng = np.random.default_rng(5)
    x, y = rng.uniform(-1, 1, (m, k)).astype(np.float32), rng.uniform(0, 1, (n, k)).astype(np.float32)
    a, b = ctx.upload(x), ctx.upload(y)
    w, size = x.astype(np.float64).sum(1), np.abs(x).sum(1, dtype=np.float64)
    for _ in range(12):
        sums, start = [None] * 2, threading.Barrier(2)

        def ask(i):
            start.wait()
            sums[i] = a.contract(None, 1)

        g = C.c_void_p()
        ctx.check(ctx.lib.dll.hgpu_capture_begin(ctx.h))
        try:
            p = a.replicate([n]).transpose([1, 0, 2]).contract(b.replicate([m]), 2)
            threads = [threading.Thread(target=ask, args=(i,)) for i in range(2)]
            [t.start() for t in threads]
            [t.join() for t in threads]
        finally:
            ctx.check(ctx.lib.dll.hgpu_capture_end(ctx.h, C.byref(g)))
        ctx.check(ctx.lib.dll.hgpu_graph_launch(g))
        ctx.sync()
        for s in sums:
            assert np.all(np.abs(s.numpy() - w) <= (2.0 ** -24 + k * 2.0 ** -53) * size)
        del p, sums, s
        ctx.check(ctx.lib.dll.hgpu_graph_destroy(g))


@pytest.mark.parametrize("t,sizes", [(8, [(128, 128)] * 3), (9, [(128, 100), (128, 128)]), (8, [(130, 96)] * 4), (7, [(128, 128)] * 3)])
def test_products_of_a_recurrence_together(host, t, sizes):
    """Weight gradients of eight and more terms that go out together take longer shares of K than each by itself, and the sums of
    their partial results, with the row sums beside them, go by the new shares."""
    rng = np.random.default_rng(t + len(sizes))
    k = 5003
    xs, ys = [], []
    for m, n in sizes:
        xs.append([rng.uniform(-1, 1, (m, k)).astype(np.float32) for _ in range(t)])
        ys.append([rng.uniform(-1, 1, (k, n)).astype(np.float32) for _ in range(t)])
    a, b = [[host.concrete(x) for x in x1] for x1 in xs], [[host.concrete(y) for y in y1] for y1 in ys]

    def program():
        products = []
        for a1, b1 in zip(a, b):
            s = a1[0].smatmul2(b1[0])
            for u, v in zip(a1[1:], b1[1:]):
                s = s + u.smatmul2(v)
            products.append(s)
        held.force(host, *products)
        total = rows(a[0][0])
        for u in a[0][1:]:
            total = total + rows(u)
        return products + [total]

    eager = [v.numpy() for v in program()]
    graph, res, labels = held.recorded(host, program)
    together = [s for s in labels if s.startswith("gemm_wide_group[")]
    assert len(together) == 1 and together[0].count("|") == len(sizes) - 1, labels
    want = [sum(x.astype(np.float64) @ y for x, y in zip(x1, y1)) for x1, y1 in zip(xs, ys)] + [sum(x.sum(1, dtype=np.float64) for x in xs[0])]
    size = [sum(np.abs(x).astype(np.float64) @ np.abs(y) for x, y in zip(x1, y1)) for x1, y1 in zip(xs, ys)] + [sum(np.abs(x).sum(1, dtype=np.float64) for x in xs[0])]
    try:
        for _ in range(3):
            graph.launch()
            host.sync()
            for got, e, w, s in zip(res, eager, want, size):
                # sixteen products to a rounded addition, and the sum of the partial results
                assert np.all(np.abs(got.numpy() - w) <= (t * k / 16 + 17) * 2.0 ** -24 * s)
                assert t >= 8 or e.ndim < 2 or np.array_equal(got.numpy(), e)      # fewer terms: the bits of the products one by one
            [v.numpy() for v in program()]
    finally:
        graph.free()

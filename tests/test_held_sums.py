"""Sums of partial results wait for one another (csrc/smallk.hip, make_way_locked; csrc/contract.hip, k_contract_group)."""
import ctypes as C

import numpy as np
import pytest

from conftest import pkg
from test_gemm_split import product

pytestmark = pytest.mark.gpu

EPS = {np.float64: 2.0 ** -53, np.float32: 2.0 ** -24}


def recorded(host, program):
    """The recorded program, its results, and how often each kernel is launched by it."""
    lib, ctx = pkg.capi.Lib(), host.dll.hh_array_ctx(host.h)
    assert lib.profile_enable(ctx, 2) == 0
    graph, res = host.capture(program)
    report = C.create_string_buffer(1 << 16)
    assert lib.profile_report(ctx, report, len(report)) == 0 and lib.profile_enable(ctx, 0) == 0
    return graph, res, {line.rsplit(None, 4)[0]: int(line.rsplit(None, 4)[1]) for line in report.value.decode().splitlines()}


def force(host, *values):
    """Submitted now, in this order (products and sums of a program are submitted when they are asked for)."""
    for v in values:
        host.check(host.dll.hh_force(host.h, v.h))


class Value:
    """A device array, what it should be and how far it may be from that."""

    def __init__(self, arr, want, bound):
        self.arr, self.want, self.bound = arr, want, bound

    def check(self):
        assert np.all(np.abs(self.arr.numpy() - self.want) <= self.bound)


def times(gpu, x, y, dt):
    """x y^T, split along its long inner dim: every product and addition rounds once at most, here and in the split into bf16 parts."""
    k = x.shape[1]
    a, b = x.astype(np.float64), y.astype(np.float64)
    return Value(product(gpu, x, y, "KK"), a @ b.T, 4 * (k + 8) * EPS[dt] * (np.abs(a) @ np.abs(b).T))


def row_sums(gpu, x, dt):
    a = x.astype(np.float64)
    return Value(gpu.upload(x).contract(None, 1), a.sum(1), 4 * x.shape[1] * EPS[dt] * np.abs(a).sum(1))


def add(v, w, dt):
    s = v.want + w.want
    return Value(v.arr.ewise2("add", w.arr), s, v.bound + w.bound + 2 * EPS[dt] * (np.abs(s) + v.bound + w.bound))


@pytest.mark.parametrize("dt", [np.float64, np.float32])
@pytest.mark.parametrize("count", [1, 2, 5, 14, 27])
def test_sums_of_many_shapes_together(gpu, dt, count):
    """More of them than one launch takes (twelve), with a few and with many partial results, whole and partly filled
    blocks of outputs; every third one is asked for while the others wait."""
    rng = np.random.default_rng(count)
    shapes = [(64, 64, 9000), (100, 37, 20000), (300, 130, 5000), (784, 300, 2000), (17, 16, 30000), (128, 128, 16411)]
    vals, asked = [], []
    for i in range(count):
        m, n, k = shapes[i % len(shapes)]
        vals.append(times(gpu, rng.uniform(-1, 1, (m, k)).astype(dt), rng.uniform(0, 1, (n, k)).astype(dt), dt))
        if i % 3 == 1:
            asked.append(add(vals[-1], vals[-1], dt))
            vals.append(row_sums(gpu, rng.uniform(-1, 1, (100, 70000)).astype(dt), dt))
    for v in asked + vals:
        v.check()


@pytest.mark.parametrize("dt", [np.float64, np.float32])
@pytest.mark.parametrize("seed", range(4))
def test_random_orders(gpu, dt, seed):
    """Products, sums of rows, additions of earlier results and writes into memory that held launches read, in any order."""
    rng = np.random.default_rng(seed)
    m, n, k = 96, 80, 6001
    xs = [rng.uniform(-1, 1, (m, k)).astype(dt) for _ in range(3)]
    ups = [gpu.upload(x) for x in xs]
    y = rng.uniform(-1, 1, (n, k)).astype(dt)
    b = gpu.upload(y)
    vals = [times(gpu, xs[0], y, dt)]
    for _ in range(40):
        what, i = rng.integers(0, 5), int(rng.integers(0, 3))
        if what < 2:
            a = xs[i].astype(np.float64)
            c = y.astype(np.float64)
            arr = ups[i].replicate([n]).transpose([1, 0, 2]).contract(b.replicate([m]), 2)
            vals.append(Value(arr, a @ c.T, 4 * (k + 8) * EPS[dt] * (np.abs(a) @ np.abs(c).T)))
        elif what == 2:
            two = [v for v in vals if v.want.ndim == 2]
            vals.append(add(two[int(rng.integers(0, len(two)))], two[-1], dt))
        elif what == 3:
            a = xs[i].astype(np.float64)
            vals.append(Value(ups[i].contract(None, 1), a.sum(1), 4 * k * EPS[dt] * np.abs(a).sum(1)))
        else:
            xs[i] = rng.uniform(-1, 1, (m, k)).astype(dt)
            ups[i].assign(gpu.upload(xs[i]))
    for v in vals:
        v.check()


def test_a_sum_into_the_callers_array_comes_after_held_reads(gpu):
    rng = np.random.default_rng(3)
    x, out = rng.uniform(-1, 1, (100, 5000)), rng.uniform(-1, 1, 100)
    a, o = gpu.upload(x), gpu.upload(out)
    before = o.replicate([3000]).contract(None, 0)          # held, reads o
    a.contract_noalloc(None, 1, o)
    np.testing.assert_allclose(before.numpy(), out.sum() * 3000, rtol=1e-10, atol=1e-9)
    np.testing.assert_allclose(o.numpy(), x.sum(1), rtol=1e-10, atol=1e-10)


def test_few_launches(gpu):
    """Three split products and two sums of rows: one launch adds up all their partial results."""
    rng = np.random.default_rng(4)
    pairs = [(gpu.upload(rng.uniform(-1, 1, (200, 8000))), gpu.upload(rng.uniform(-1, 1, (100, 8000)))) for _ in range(3)]
    wide = gpu.upload(rng.uniform(-1, 1, (128, 140000)))
    gpu.check(gpu.lib.profile_enable(gpu.h, 2))
    out = [a.replicate([100]).transpose([1, 0, 2]).contract(b.replicate([200]), 2) for a, b in pairs] + [wide.contract(None, 1) for _ in range(2)]
    out[0].numpy()
    labels = list(gpu.profile_report())
    gpu.check(gpu.lib.profile_enable(gpu.h, 0))
    assert sum(s.startswith("contract_group") or s.startswith("gemm_sum_partials") for s in labels) == 1, labels


@pytest.mark.parametrize("dt", [np.float64, np.float32])
@pytest.mark.parametrize("n", [37, 128])
@pytest.mark.parametrize("order", [(0, 1), (1, 0), (1, 2, 0), (0, 2), (1, 2)])
def test_sums_of_products_of_several_layouts(gpu, dt, n, order):
    """A product over k, a row's sum times one element that every column repeats, a column's repeated down the rows."""
    rng = np.random.default_rng(n)
    m, k = 130, 3001
    x, y = rng.uniform(-1, 1, (m, k)).astype(dt), rng.uniform(-1, 1, (n, k)).astype(dt)
    c = np.asarray(0.75, dt)
    a = gpu.upload(x).replicate([n]).transpose([1, 0, 2])
    b = gpu.upload(y).replicate([m])
    one = gpu.upload(c).replicate([m, n, k])
    a64, b64 = x.astype(np.float64), y.astype(np.float64)
    pairs = [(a, b), (a, one), (one, b)]
    want = [a64 @ b64.T, np.broadcast_to(0.75 * a64.sum(1)[:, None], (m, n)), np.broadcast_to(0.75 * b64.sum(1)[None, :], (m, n))]
    size = [np.abs(a64) @ np.abs(b64).T, 0.75 * np.abs(a64).sum(1)[:, None] + np.zeros((m, n)), 0.75 * np.abs(b64).sum(1)[None, :] + np.zeros((m, n))]
    got = gpu.contract_sum([pairs[i] for i in order], 2).numpy()
    bound = 4 * (k + 8) * EPS[dt] * sum(size[i] for i in order)
    assert np.all(np.abs(got - sum(want[i] for i in order)) <= bound)


@pytest.mark.parametrize("dt", [np.float64, np.float32])
@pytest.mark.parametrize("p,q,k", [(784, 128, 1000), (783, 127, 601), (500, 33, 1024), (96, 100, 1023)])
def test_bare_products_with_k_shared_out(gpu, dt, p, q, k):
    """Few tiles under a long K: whole partial results, tiles with one row or column among them."""
    rng = np.random.default_rng(k)
    vals = [times(gpu, rng.uniform(-1, 1, (q, k)).astype(dt), rng.uniform(-1, 1, (p, k)).astype(dt), dt) for _ in range(2)]
    for v in vals:
        v.check()


@pytest.fixture(scope="module")
def host():
    return pkg.hostapi.Host()


@pytest.mark.parametrize("dt", [np.float64, np.float32])
@pytest.mark.parametrize("shapes", [
    [(128, 128, 30000)] * 3,                                        # as many blocks each: they take turns
    [(128, 128, 30000), (129, 128, 30000)],                         # a tile row more
    [(300, 784, 5000), (100, 300, 5000), (120, 100, 9001)],         # one after the other
    [(130, 100, 20000)] * 5 + [(96, 96, 20011)],                    # more than one launch takes
    [(1000, 300, 1100)],
])
@pytest.mark.parametrize("lay", ["KK", "RK", "KR", "RR"])
def test_products_of_a_recording_go_out_together(host, dt, shapes, lay):
    """Weight gradients, the first operand shared where sizes agree: every replay is what the products submitted one by one
    give, bit for bit, and within rounding of numpy."""
    rng = np.random.default_rng(len(shapes))
    shared, pairs = {}, []
    for m, n, k in shapes:
        if (m, k) not in shared:
            shared[m, k] = rng.uniform(-1, 1, (m, k)).astype(dt)
        pairs.append((shared[m, k], rng.uniform(0, 1, (n, k)).astype(dt)))
    up = {}

    def put(x, how):
        key = (id(x), how)
        if key not in up:
            up[key] = host.concrete(x) if how == "K" else host.concrete(np.ascontiguousarray(x.T)).stranspose([1, 0])
        return up[key]

    ops = [(put(x, lay[0]), put(y, lay[1]).stranspose([1, 0])) for x, y in pairs]

    def program():
        out = [a.smatmul2(b) for a, b in ops]
        return out + [a.stranspose([1, 0]).ssum() for a, _ in ops[:2]]

    eager = [v.numpy() for v in program()]
    graph, res, labels = recorded(host, program)
    # (products of one layout, a launch takes four of them)
    alike = len(pairs) if dt == np.float64 or min(min(m, n) for m, n, _ in shapes) > 32 else sum(min(m, n) <= 32 for m, n, _ in shapes)
    assert alike < 2 or sum(k.count("|gemm_f") * v for k, v in labels.items() if k.startswith("gemm_wide_group[")) >= (alike + 1) // 2, labels
    try:
        for _ in range(3):
            graph.launch()
            host.sync()
            for got, want in zip(res, eager):
                assert np.array_equal(got.numpy(), want)
            [v.numpy() for v in program()]
    finally:
        graph.free()
    for (x, y), got in zip(pairs, eager):
        a, b = x.astype(np.float64), y.astype(np.float64)
        assert np.all(np.abs(got - a @ b.T) <= 4 * (x.shape[1] + 8) * EPS[dt] * (np.abs(a) @ np.abs(b).T))


@pytest.mark.parametrize("dt", [np.float64, np.float32, np.int8, np.int64])
@pytest.mark.parametrize("rows,n", [(1, 16384), (3, 16385), (1, 50000), (16, 40961), (2, 300001)])
def test_extrema_of_long_rows(gpu, dt, rows, n):
    """Pieces of a row to many blocks, the last of which picks: again and again, ties to the first."""
    rng = np.random.default_rng(n)
    x = rng.integers(-100, 100, (rows, n)).astype(dt)
    x[:, n // 2] = x[:, n - 1] = 101
    a = gpu.upload(x)
    for _ in range(4):
        assert np.array_equal(a.argminmax_last(True).numpy(), x.argmax(1))
        assert np.array_equal(a.argminmax_last(False).numpy(), x.argmin(1))
    if dt in (np.float64, np.float32):
        x[0, 7] = np.inf
        x[-1, n - 3] = -np.inf
        a = gpu.upload(x)
        assert np.array_equal(a.argminmax_last(True).numpy(), x.argmax(1))
        assert np.array_equal(a.argminmax_last(False).numpy(), x.argmin(1))


@pytest.mark.parametrize("dt", [np.float64, np.float32])
@pytest.mark.parametrize("rows,n", [(128, 4200), (17, 30000), (300, 2000), (1, 9000)])
def test_row_sums_in_chunks_wait(host, dt, rows, n):
    """Both stages of a sum in chunks, the negation of a result, and a result read on the way, recorded and not."""
    rng = np.random.default_rng(rows)
    x, y = (rng.uniform(-1, 1, (28, rows, n // 28)).astype(dt) for _ in range(2))
    a, b = host.concrete(x), host.concrete(y)

    def program():
        s, t = (v.stranspose([1, 0, 2]).sreshape((rows, 28 * (n // 28))).stranspose([1, 0]).ssum() for v in (a, b))
        return [s, -t, s + t, -(a.ssum0())]

    want = [x.astype(np.float64).sum((0, 2)), -y.astype(np.float64).sum((0, 2)), (x.astype(np.float64) + y).sum((0, 2)), -x.astype(np.float64).sum()]
    size = [np.abs(x).sum((0, 2)), np.abs(y).sum((0, 2)), (np.abs(x) + np.abs(y)).sum((0, 2)), np.abs(x).sum()]
    eager = [v.numpy() for v in program()]
    graph, res = host.capture(program)
    try:
        for _ in range(3):
            graph.launch()
            host.sync()
            for got, e in zip(res, eager):
                assert np.array_equal(got.numpy(), e)
            [v.numpy() for v in program()]
    finally:
        graph.free()
    for e, w, m in zip(eager, want, size):      # sums run in doubles: their roundings, and those to the result's type and of the addition
        assert np.all(np.abs(e - w) <= 4 * (EPS[dt] + n * EPS[np.float64]) * m)


@pytest.mark.parametrize("dt", [np.float64, np.float32])
def test_programs_over_a_few_elements(host, dt):
    """What an objective ends with: one and two operands, still and moving, sums of theirs read at once and later."""
    rng = np.random.default_rng(5)
    x, c = rng.uniform(-1, 1, (64, 4001)).astype(dt), np.asarray(0.37, dt)
    a, k = host.concrete(x), host.concrete(c)

    def program():
        s = a.stranspose([1, 0]).ssum()
        t = a.ssum0()
        return [-(t * k), (t - k) * t, -s, s * k.sreplicate0N((64,)) - s, (-(t * k)) + k]

    x, k64, e = x.astype(np.float64), float(c), EPS[dt]
    s, t, ms, mt = x.sum(1), x.sum(), np.abs(x).sum(1), np.abs(x).sum()
    want = [(-(t * k64), mt), ((t - k64) * t, 2 * (mt + 1) * mt), (-s, ms), (s * k64 - s, 2 * ms), (-(t * k64) + k64, mt + 1)]
    eager = [v.numpy() for v in program()]
    for got, (w, m) in zip(eager, want):         # 64-bit sums, one rounding to the type, one per operation
        assert np.all(np.abs(got - w) <= 8 * (e + 70000 * EPS[np.float64]) * m)
    graph, res = host.capture(program)
    try:
        for _ in range(3):
            graph.launch()
            host.sync()
            assert all(np.array_equal(r.numpy(), v) for r, v in zip(res, eager))
            [v.numpy() for v in program()]
    finally:
        graph.free()


@pytest.mark.parametrize("n", [64, 65, 1000, 2500, 4095, 4096, 100003])
@pytest.mark.parametrize("with_pass", [False, True])
def test_dot_products_of_expressions_round_once(host, n, with_pass):
    """fp32: neighbouring products cancel but for what rounding them to fp32 would leave; summed alone, and in the pass that writes
    another expression of this shape."""
    rng = np.random.default_rng(n)
    x, y = (rng.uniform(0.5, 1, n).astype(np.float32) for _ in range(2))
    y[1::2] = -(x[0:n - 1:2] * y[0:n - 1:2] / x[1::2])
    y[n // 2 * 2:] = 0
    a, b = host.concrete(x), host.concrete(y)

    e = -a
    s = e.sdot0(b)
    if with_pass:
        assert np.array_equal((e * b).numpy(), -x * y)
    p = x.astype(np.float64) * y
    assert abs(float(s.numpy()) + p.sum()) <= 2.0 ** -24 * abs(p.sum()) + n * 2.0 ** -52 * np.abs(p).sum()


@pytest.mark.parametrize("terms", [9, 15, 16, 23, 24, 31, 32])
def test_partial_results_are_added_in_short_chains(gpu, terms):
    """One partial result of 1 and others of a quarter of its last place: of eight chains the one that has the 1 loses the others of its
    own, and the chains meet in three roundings."""
    m, k = 300, 64
    pairs = []
    for t in range(terms):
        x, y = np.zeros((m, k), np.float32), np.zeros((m, k), np.float32)
        x[:, t], y[:, t] = 1 if t == 0 else 2.0 ** -25, 1
        pairs.append((gpu.upload(x).replicate([m]).transpose([1, 0, 2]), gpu.upload(y).replicate([m])))
    gpu.profile(2)
    got = gpu.contract_sum(pairs, 2).numpy().astype(np.float64)
    labels = list(gpu.profile_report())
    gpu.profile(0)
    assert any("s%d," % terms in s for s in labels) and "gemm_sum_partials" in labels, labels
    want = 1 + (terms - 1) * 2.0 ** -25
    assert np.all(np.abs(got - want) <= (terms - 1) // 8 * 2.0 ** -25 + 3 * 2.0 ** -24), np.unique((got - want) * 2 ** 24)


def test_memory_of_held_work_comes_back_for_an_allocation(gpu):
    """Sums that wait keep the arrays they read, which nobody else has any more: a request that the device cannot serve sends them out."""
    x = gpu.upload(np.ones((200, 100003), np.float32))
    big = x.ewise1("neg")                                  # (blocks of this size exist, and none is left)
    try:
        gpu.check(gpu.lib.inject_alloc_failure(gpu.h, 1))      # for the sums
        s = big.slice(0, 0, 100).slice(1, 0, 4096).contract(None, 1)
        del big                                            # only the held sum has it now
        y = x.ewise1("neg")
    finally:
        gpu.check(gpu.lib.inject_alloc_failure(gpu.h, -1))
    assert np.array_equal(s.numpy(), np.full(100, -4096, np.float32)) and y.numpy()[0, 0] == -1


def test_held_work_keeps_a_bounded_amount_of_memory(gpu):
    """Sums of small parts of large arrays that are released at once."""
    fresh = pkg.capi.Lib().context(0)
    n = 1 << 27                                            # 512 MB
    x = fresh.upload(np.zeros(1, np.float32)).replicate([n]).reshape([n])
    before = fresh.mem_stats()[1]
    sums = []
    for _ in range(24):
        big = x.ewise1("cos")
        sums.append(big.slice(0, 0, 100 * 4096).reshape([100, 4096]).contract(None, 1))
        del big
    assert fresh.mem_stats()[1] - before <= 6 << 30
    for s in sums:
        assert np.array_equal(s.numpy(), np.full(100, 4096, np.float32))
    del x, sums, s
    fresh.shutdown()


def test_a_recording_takes_the_memory_it_has(gpu):
    """Inside a recording blocks cannot be freed: held work goes out, and a larger block serves where none of the size is left."""
    ctx = pkg.capi.Lib().context(0)
    dll = ctx.lib.dll
    x = np.random.default_rng(1).uniform(-1, 1, (300, 20000)).astype(np.float32)
    ctx.check(ctx.lib.inject_alloc_failure(ctx.h, 4))      # for the two arrays here, and the first two below
    a, large = ctx.upload(x), ctx.upload(np.zeros(200 << 20, np.int8))
    ctx.sync()
    del large
    ctx.check(dll.hgpu_capture_begin(ctx.h))
    try:
        neg = a.ewise1("neg")
        s = neg.slice(1, 0, 4096).contract(None, 1)        # waits
        del neg
        y = a.ewise1("abs")                                # the block of neg, which the sum had
        z = a.ewise1("neg")                                # the large one
    finally:
        g = C.c_void_p()
        ctx.check(dll.hgpu_capture_end(ctx.h, C.byref(g)))
    ctx.check(ctx.lib.inject_alloc_failure(ctx.h, -1))
    for _ in range(2):
        ctx.check(dll.hgpu_graph_launch(g))
        ctx.sync()
        want = -x[:, :4096].astype(np.float64).sum(1)
        assert np.array_equal(y.numpy(), np.abs(x)) and np.array_equal(z.numpy(), -x)
        assert np.all(np.abs(s.numpy() - want) <= 2.0 ** -24 * np.abs(want) + 2.0 ** -40)
    ctx.check(dll.hgpu_graph_destroy(g))


def test_the_end_of_an_objective_waits_in_recordings_only(host, gpu):
    """`negate sum * c` joins the last sums of a recording; submitted one by one it is a launch of its own, which goes out at once."""
    prog = [(0, pkg.capi.OP1["neg"], 0, 0, 0, 0), (1, pkg.capi.OP2["mul"], 0, 2, 1, 0)]
    ins = [gpu.upload(np.asarray(v, np.float32)) for v in (3.0, 0.5)]
    x = gpu.upload(np.ones((100, 5000), np.float32))
    gpu.profile(2)
    s = x.contract(None, 1)                                # waits
    got = [gpu.fused_map(ins, prog, [3])[0] for _ in range(2)]
    labels = gpu.profile_report()
    gpu.profile(0)
    assert labels["tiny_map"][0] == 2 and not any("|" in k for k in labels), labels
    assert [float(v.numpy()) for v in got] == [-1.5, -1.5] and np.array_equal(s.numpy(), np.full(100, 5000, np.float32))
    x = host.concrete(np.random.default_rng(1).uniform(-1, 1, (100, 5000)).astype(np.float32))
    c = host.concrete(np.asarray(0.25, np.float32))

    def program():
        s = x.ssum0()
        force(host, s)
        return [-s * c, x.stranspose([1, 0]).ssum()]

    eager = [v.numpy() for v in program()]
    graph, res, labels = recorded(host, program)
    try:
        assert any("tiny_map" in k for k in labels), labels
        for _ in range(3):
            graph.launch()
            host.sync()
            assert all(np.array_equal(r.numpy(), e) for r, e in zip(res, eager))
            [v.numpy() for v in program()]
    finally:
        graph.free()


def test_sums_that_nobody_reads_do_not_gather(gpu):
    """Submitted one by one, pass after pass: what is held goes out after a few launches that did not need it."""
    fresh = pkg.capi.Lib().context(0)
    x = fresh.upload(np.ones((100, 100003), np.float32))   # 40 MB
    sums, size = [], fresh.mem_stats()[1]
    for _ in range(48):
        big = x.ewise1("neg")
        sums.append(big.slice(1, 0, 4096).contract(None, 1))
        del big
    assert fresh.mem_stats()[1] - size <= 12 * (41 << 20)
    for s in sums:
        assert np.array_equal(s.numpy(), np.full(100, -4096, np.float32))
    del x, sums, s
    fresh.shutdown()

"""Held-back products that read one another's results column by column run as one kernel (csrc/smallk_chain.hpp): the
steps of an unrolled recurrence and of its transposition.  Every step is compared with numpy on the results that the
device itself gave for the steps before, so that the bound is that of one step."""
import numpy as np
import pytest

from conftest import capi
from test_contract_sum_map import matmul_views

pytestmark = pytest.mark.gpu

O1, O2, CMP = capi.OP1, capi.OP2, capi.CMP


def chains(ctx, work):
    """(what `work` gives, how many chains were launched)"""
    ctx.check(ctx.lib.profile_enable(ctx.h, 2))
    out = work()
    labels = ctx.profile_report()
    ctx.check(ctx.lib.profile_enable(ctx.h, 0))
    return out, sum(v[0] for k, v in labels.items() if "[chain:" in k), labels


def step_bound(dt, ks):
    # |w| <= 0.3, |x|, |h| <= 1: a rounding per product and per addition, and a program with a few units of its own
    return np.finfo(dt).eps * (0.3 * sum(ks) * (sum(ks) + 8) + 8)


@pytest.mark.parametrize("dt", [np.float64, np.float32])
@pytest.mark.parametrize("width,batch,k_in,steps,layers", [
    (128, 150, 28, 9, 2),       # four columns a block, the weights partly in LDS (fp64)
    (128, 1000, 28, 8, 2),      # the fewest levels: 8 of one layer and one more
    (64, 1021, 17, 12, 2),      # columns that fill no group of four; k of no whole tile
    (64, 2053, 28, 8, 2),       # more columns a block, a ragged last block
    (17, 4100, 30, 9, 2),       # two row groups, the second one row high
    (130, 260, 5, 8, 1),        # one layer: all wavefronts on it, the ninth row group is one wavefront's
    (16, 5000, 28, 10, 1),      # one row group, 20 columns a block
    (40, 700, 48, 9, 3),        # three layers: four, two and two wavefronts
    (100, 515, 33, 8, 2),
    # fp64 by lone columns, one and two to a block
    (128, 256, 28, 8, 2),       # a block for every CU
    (128, 511, 28, 8, 2),       # two columns, the last block has one
    (100, 257, 33, 8, 2),       # a wavefront with one row group beside those with two
    (130, 200, 5, 8, 1),        # one layer
    (17, 131, 30, 9, 2),        # the second row group one row high
    (40, 61, 70, 9, 3),         # k of no whole 64, three layers
    (64, 512, 17, 8, 2),        # two columns with one row group a wavefront: in groups of four
])
def test_recurrence_forward(gpu, dt, width, batch, k_in, steps, layers):
    rng = np.random.default_rng(width + batch)
    kin = [k_in] + [width] * (layers - 1)
    wx = [rng.uniform(-0.3, 0.3, (width, kin[l])).astype(dt) for l in range(layers)]
    wh = [rng.uniform(-0.3, 0.3, (width, width)).astype(dt) for _ in range(layers)]
    bs = [rng.uniform(-0.5, 0.5, (width,)).astype(dt) for _ in range(layers)]
    xs = [rng.uniform(-1, 1, (k_in, batch)).astype(dt) for _ in range(steps)]
    wo = rng.uniform(-0.3, 0.3, (10, width)).astype(dt)
    prog = [(1, O2["add"], 0, 0, 1, 0), (0, O1["tanh"], 0, 2, 0, 0)]

    def work():
        up = gpu.upload
        zero = up(np.zeros((), dt)).replicate([batch]).replicate([width])
        params = [(up(wx[l]), up(wh[l]), up(bs[l]).replicate([batch]).transpose([1, 0])) for l in range(layers)]
        last, no_bias, xa = up(wo), up(np.zeros((10,), dt)).replicate([batch]).transpose([1, 0]), [up(x) for x in xs]
        hs = []
        for l in range(layers):       # layer by layer (an upload would send out what is held back)
            (w, v, b), h = params[l], []
            for t in range(steps):
                x = xa[t] if l == 0 else hs[l - 1][t]
                h.append(gpu.contract_sum_map([matmul_views(w, x), matmul_views(v, h[-1] if h else zero)], 2, [None, b], prog, [3])[0])
            hs.append(h)
        # a readout, and where it is negative (a result of another type)
        out = gpu.contract_sum_map([matmul_views(last, hs[-1][-1])], 2, [None, no_bias], [(2, CMP["lt"], 0, 0, 1, 0)], [0, 2])
        return [[a.numpy() for a in h] for h in hs], [a.numpy() for a in out]

    (hs, out), n, labels = chains(gpu, work)
    assert n == 1, labels
    if dt == np.float64 and layers > 1:      # lone columns where one or two to each of 256 CUs are enough
        lone = 1 if batch <= 256 else 2 if batch <= 512 and width > 64 else None
        assert any(",t%d]" % lone in k for k in labels) if lone else not any(",t1]" in k or ",t2]" in k for k in labels), labels
    for l in range(layers):
        for t in range(steps):
            x = (xs[t] if l == 0 else hs[l - 1][t]).astype(np.float64)
            s = hs[l][t - 1].astype(np.float64) if t else np.zeros((width, batch))
            want = np.tanh(wx[l].astype(np.float64) @ x + wh[l].astype(np.float64) @ s + bs[l].astype(np.float64)[:, None])
            assert hs[l][t].dtype == dt and np.max(np.abs(hs[l][t] - want)) <= step_bound(dt, [kin[l], width]), (l, t)
    want = wo.astype(np.float64) @ hs[-1][-1].astype(np.float64)
    assert np.max(np.abs(out[0] - want)) <= step_bound(dt, [width])
    assert np.array_equal(out[1], out[0] < 0)
    (again, _), _, _ = chains(gpu, work)
    for a, b in zip(sum(again, []), sum(hs, [])):
        assert np.array_equal(a, b)


@pytest.mark.parametrize("dt", [np.float64, np.float32])
@pytest.mark.parametrize("width,batch,steps", [(128, 150, 9), (48, 1030, 10), (40, 701, 10), (100, 250, 9), (72, 203, 10), (128, 301, 9)])
def test_recurrence_backward(gpu, dt, width, batch, steps):
    """d2_t = (V2^T d2_(t+1)) * (1 - h2_t^2) + d2_(t+1), d1_t = (W2^T d2_t + V1^T d1_(t+1)) * (1 - h1_t^2): weights transposed,
    whole arrays as inputs of the program, among them a result of the chain."""
    rng = np.random.default_rng(width * steps)
    v2, w2, v1, wo = (rng.uniform(-0.3, 0.3, s).astype(dt) / dt(4) for s in ((width, width), (width, width), (width, width), (10, width)))
    h1, h2 = ([rng.uniform(-1, 1, (width, batch)).astype(dt) for _ in range(steps)] for _ in range(2))
    dl = rng.uniform(-1, 1, (10, batch)).astype(dt)
    # (sum) * (h - h * h)
    prog = [(1, O2["mul"], 0, 1, 1, 0), (1, O2["sub"], 0, 1, 2, 0), (1, O2["mul"], 0, 0, 3, 0)]
    prog_plus = [(1, O2["mul"], 0, 1, 1, 0), (1, O2["sub"], 0, 1, 3, 0), (1, O2["mul"], 0, 0, 4, 0), (1, O2["add"], 0, 5, 2, 0)]

    def work():
        up = gpu.upload
        tr = {k: up(v).transpose([1, 0]) for k, v in (("v2", v2), ("w2", w2), ("v1", v1), ("wo", wo))}
        a1, a2, adl = [up(h) for h in h1], [up(h) for h in h2], up(dl)
        d2, d1 = [None] * steps, [None] * steps
        for t in reversed(range(steps)):
            if t == steps - 1:
                d2[t] = gpu.contract_sum_map([matmul_views(tr["wo"], adl)], 2, [None, a2[t]], prog, [4])[0]
            else:
                d2[t] = gpu.contract_sum_map([matmul_views(tr["v2"], d2[t + 1])], 2, [None, a2[t], d2[t + 1]], prog_plus, [6])[0]
        for t in reversed(range(steps)):
            terms = [matmul_views(tr["w2"], d2[t])] + ([matmul_views(tr["v1"], d1[t + 1])] if t < steps - 1 else [])
            d1[t] = gpu.contract_sum_map(terms, 2, [None, a1[t]], prog, [4])[0]
        return [a.numpy() for a in d2], [a.numpy() for a in d1]

    (d2, d1), n, labels = chains(gpu, work)
    assert n == 1, labels
    f = lambda a: a.astype(np.float64)
    # a step's values are bounded by the numbers themselves: relative to the largest magnitude summed
    for t in range(steps):
        src, w = (dl, wo) if t == steps - 1 else (d2[t + 1], v2)
        g = f(h2[t]) - f(h2[t]) ** 2
        want = (f(w).T @ f(src)) * g + (0 if t == steps - 1 else f(d2[t + 1]))
        mag = (np.abs(f(w)).T @ np.abs(f(src))) * 2 + (0 if t == steps - 1 else np.abs(f(d2[t + 1])))
        assert np.all(np.abs(d2[t] - want) <= np.finfo(dt).eps * (width + 12) * mag), t
        want, mag = f(w2).T @ f(d2[t]), np.abs(f(w2)).T @ np.abs(f(d2[t]))
        if t < steps - 1:
            want, mag = want + f(v1).T @ f(d1[t + 1]), mag + np.abs(f(v1)).T @ np.abs(f(d1[t + 1]))
        g = f(h1[t]) - f(h1[t]) ** 2
        assert np.all(np.abs(d1[t] - want * g) <= np.finfo(dt).eps * (2 * width + 12) * mag * 2), t


@pytest.mark.parametrize("dt", [np.float64, np.float32])
def test_what_breaks_a_chain(gpu, dt):
    """A step that reads a result as the weights, or shifted by a column, is no part of the chain: it and what follows from
    it run by themselves, after the chain, with the right values."""
    rng = np.random.default_rng(5)
    n, steps = 128, 12
    w = rng.uniform(-0.1, 0.1, (n, n)).astype(dt)
    x = rng.uniform(-1, 1, (n, n)).astype(dt)
    prog = [(0, O1["tanh"], 0, 0, 0, 0)]

    def work(break_at, how):
        wa, h, xa, res = gpu.upload(w), gpu.upload(x), gpu.upload(x), []
        for t in range(steps):
            if t == break_at and how == "weights":
                pair = matmul_views(h, xa)
            elif t == break_at:
                pair = matmul_views(wa, h.reverse(1))
            else:
                pair = matmul_views(wa, h)
            h = gpu.contract_sum_map([pair], 2, [None], prog, [1])[0]
            res.append(h)
        return [a.numpy() for a in res]

    for break_at, how in ((9, "weights"), (9, "columns"), (2, "weights")):
        got, k, labels = chains(gpu, lambda: work(break_at, how))
        assert k == (1 if break_at >= 8 else 0), labels
        prev = x.astype(np.float64)
        for t, g in enumerate(got):
            if t == break_at and how == "weights":
                want = prev @ x.astype(np.float64)
            elif t == break_at:
                want = w.astype(np.float64) @ prev[:, ::-1]
            else:
                want = w.astype(np.float64) @ prev
            assert np.max(np.abs(g - np.tanh(want))) <= step_bound(dt, [n]) * 4, (how, t)
            prev = g.astype(np.float64)


@pytest.mark.parametrize("dt", [np.float32, np.float64])
def test_values_that_are_no_numbers_stay_in_their_column(gpu, dt):
    """Infinities and NaN in some columns of the input reach the results of those columns only."""
    rng = np.random.default_rng(6)
    n, b, steps = 80, 203, 9
    w = rng.uniform(-0.3, 0.3, (n, n)).astype(dt)
    x = rng.uniform(-1, 1, (n, b)).astype(dt)
    x[3, 7], x[79, 100], x[0, 202] = np.inf, np.nan, -np.inf
    wa, h = gpu.upload(w), gpu.upload(x)

    def work(h):
        for _ in range(steps):
            h = gpu.contract_sum_map([matmul_views(wa, h)], 2, [None], [(0, O1["neg"], 0, 0, 0, 0)], [1])[0]
        return h.numpy()

    got, k, labels = chains(gpu, lambda: work(h))
    assert k == 1, labels
    bad = np.zeros(b, bool)
    bad[[7, 100, 202]] = True
    assert np.all(np.isfinite(got[:, ~bad])) and np.all(np.isnan(got[:, bad]))


@pytest.mark.parametrize("dt", [np.float64, np.float32])
def test_a_chain_longer_than_a_kernels_arguments(gpu, dt):
    """h_t = tanh (W x_t + V h_(t-1) + e_t) over 150 steps, three arrays a step: a second kernel goes on where the first one's pointers end,
    with the last result of the first read as an array."""
    rng = np.random.default_rng(11)
    width, batch, steps = 64, 96, 150
    w, v = (rng.uniform(-0.3, 0.3, (width, width)).astype(dt) for _ in range(2))
    xs, es = ([rng.uniform(-1, 1, (width, batch)).astype(dt) for _ in range(steps)] for _ in range(2))
    prog = [(1, O2["add"], 0, 0, 1, 0), (0, O1["tanh"], 0, 2, 0, 0)]

    def work():
        up = gpu.upload
        wa, va, h, xa, ea, res = up(w), up(v), up(np.zeros((), dt)).replicate([batch]).replicate([width]), [up(x) for x in xs], [up(e) for e in es], []
        for t in range(steps):
            h = gpu.contract_sum_map([matmul_views(wa, xa[t]), matmul_views(va, h)], 2, [None, ea[t]], prog, [3])[0]
            res.append(h)
        return [a.numpy().astype(np.float64) for a in res]

    got, n, labels = chains(gpu, work)
    assert n == 2, labels
    prev = np.zeros((width, batch))
    for t in range(steps):
        want = np.tanh(w.astype(np.float64) @ xs[t] + v.astype(np.float64) @ prev + es[t])
        assert np.max(np.abs(got[t] - want)) <= step_bound(dt, [width, width]), t
        prev = got[t]

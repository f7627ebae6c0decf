"""Gathers that wait, and their sum of products with an array without being written (GPU only).

The sums are formed in double: they are held to the exact sum (math.fsum of exact products) within one rounding of the element
type and n 2^-53 of the sum of magnitudes."""
import math

import numpy as np
import pytest

from conftest import capi, pkg

H = pkg.hostapi
pytestmark = pytest.mark.gpu


def gathered(t, ixs):
    ok = np.ones(ixs[0].shape, bool)
    for k, i in enumerate(ixs):
        ok &= (i >= 0) & (i < t.shape[k])
    safe = tuple(np.where(ok, i, 0) for i in ixs)
    return np.where(ok.reshape(ok.shape + (1,) * (t.ndim - len(ixs))), t[safe], 0).astype(t.dtype)


def check_dot(got, x, y):
    p = x.astype(np.longdouble) * y.astype(np.longdouble)
    exact = math.fsum(float(v) for v in p.ravel()) if x.dtype == np.float32 else float(p.sum())
    bound = np.finfo(x.dtype).eps * abs(exact) + (x.size + 8) * 2.0 ** -53 * float(np.abs(p).sum())
    assert abs(float(got) - exact) <= bound, (float(got), exact, bound)


def launches(gpu):
    return {k: v[0] for k, v in gpu.profile_report().items()}


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("rows,width,picks", [(1, 1, 1), (7, 1, 64), (50, 2, 63), (50, 3, 257), (9, 4, 65), (300, 5, 1000), (64, 128, 500), (33, 130, 77), (2000, 36, 20000)])
def test_dot_of_a_gather(gpu, dtype, rows, width, picks):
    rng = np.random.default_rng(rows + width)
    t = rng.uniform(-1, 1, (rows, width)).astype(dtype)
    ix = rng.integers(-1, rows + 1, picks)                  # some positions read zeros
    y = rng.uniform(-1, 1, (picks, width)).astype(dtype)
    want = gathered(t, [ix])
    gt, gix, gy = gpu.upload(t), gpu.upload(ix), gpu.upload(y)
    gpu.profile(True)
    for swap in (False, True):
        g = gpu.gather(gt, [gix], (picks,))
        r = gy.contract(g, 0) if swap else g.contract(gy, 0)
        del g
        check_dot(r.numpy(), want, y)
    ran = launches(gpu)
    gpu.profile(False)
    assert ran.get("gather_dot") == 2 and "gather" not in ran, ran
    # the same gather, still wanted by somebody: dot and array
    g = gpu.gather(gt, [gix], (picks,))
    r = g.contract(gy, 0)
    assert np.array_equal(g.numpy(), want)
    check_dot(r.numpy(), want, y)
    check_dot(g.contract(gy, 0).numpy(), want, y)           # written by now: the plain contraction
    both = gpu.gather(gt, [gix], (picks,))
    check_dot(both.contract(both, 0).numpy(), want, want)


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
def test_views_and_two_indices(gpu, dtype):
    """Tables and operands that start off a 16-byte boundary, a reversed table, two index arrays, one of them replicated."""
    rng = np.random.default_rng(3)
    t = rng.uniform(-1, 1, (6, 11, 9)).astype(dtype)
    i, j = rng.integers(-1, 7, (40, 5)), rng.integers(0, 11, 5)
    y = rng.uniform(-1, 1, (40, 5, 9)).astype(dtype)
    gy = gpu.upload(np.concatenate([np.zeros(1, dtype), y.ravel()])).slice(0, 1, y.size).reshape(y.shape)
    gi, gj = gpu.upload(i), gpu.upload(j).replicate([40])
    jj = np.broadcast_to(j, (40, 5))
    for table, gt in ((t, gpu.upload(t)), (t[::-1], gpu.upload(t).reverse(0)), (t[1:], gpu.upload(t).slice(0, 1, 5)),
                      (t[:, :, 1:5], gpu.upload(t).slice(2, 1, 4)), (t[:, :, ::-1], gpu.upload(t).reverse(2))):
        want = gathered(np.ascontiguousarray(table), [i, jj])
        w = want.shape[2]
        g = gpu.gather(gt, [gi, gj], (40, 5))
        check_dot(g.contract(gpu.upload(np.ascontiguousarray(y[:, :, :w])), 0).numpy(), want, y[:, :, :w])
        if w == 9:
            check_dot(g.contract(gy, 0).numpy(), want, y)
        assert np.array_equal(g.numpy(), want)


def test_positions_out_of_bounds_multiply_zeros(gpu):
    t = np.ones((4, 8))
    y = np.ones((3, 8))
    y[1, 2] = np.inf
    ix = np.array([0, 9, 2])
    g = gpu.gather(gpu.upload(t), [gpu.upload(ix)], (3,))
    assert np.isnan(float(g.contract(gpu.upload(y), 0).numpy()))
    ix[1] = 3
    g = gpu.gather(gpu.upload(t), [gpu.upload(ix)], (3,))
    assert float(g.contract(gpu.upload(y), 0).numpy()) == np.inf


def test_a_waiting_gather_reads_the_table_as_it_was():
    """Writes into the table's memory come after the gathers that wait: an overwrite, a copy, a recorded step's replay."""
    host = H.Host()
    rng = np.random.default_rng(5)
    t, ix, y = rng.uniform(-1, 1, (30, 16)), rng.integers(0, 30, 100), rng.uniform(-1, 1, (100, 16))
    table, gix, gy = host.concrete(t), host.concrete(ix), host.concrete(y)

    def pick():
        return table.sgather((100,), lambda i: [gix.sindex0([i])])
    first = pick()
    table.overwrite(t * 2)
    second = pick()
    dot = (second * gy).ssum0()
    table.assign(host.concrete(t * 3) * 1.0)
    third = pick()
    fourth = pick()
    fifth = pick()
    sixth = pick()                                           # more of them than wait at a time
    assert np.array_equal(first.numpy(), t[ix])
    check_dot(dot.numpy(), (2 * t)[ix], y)
    assert np.array_equal(second.numpy(), (2 * t)[ix])
    for g in (third, fourth, fifth, sixth):
        assert np.array_equal(g.numpy(), (t * 3)[ix])
    # a gather of a gather, and reads by an elementwise pass and a scatter
    inner = pick()
    outer = inner.sgather((50,), lambda i: [i * 2])
    gz = host.concrete(rng.integers(0, 100, 40))
    outer2 = inner.sgather((40,), lambda i: [gz.sindex0([i])])
    assert np.array_equal(outer.numpy(), (t * 3)[ix][::2])
    assert np.array_equal(outer2.numpy(), (t * 3)[ix][gz.numpy()])
    assert np.array_equal((pick() * 2.0 + 1.0).numpy(), (t * 3)[ix] * 2.0 + 1.0)
    cells = host.concrete(np.arange(100)[::-1].copy())
    assert np.array_equal(pick().sscatter(1, (100,), lambda i: [cells.sindex0([i])]).numpy(), (t * 3)[ix][::-1])


def test_dot_in_a_recording():
    host = H.Host()
    rng = np.random.default_rng(6)
    t, ix, y = rng.uniform(-1, 1, (300, 24)), rng.integers(0, 300, 5000), rng.uniform(-1, 1, (5000, 24))
    table, gix, gy = host.param(t), host.concrete(ix), host.concrete(y)

    def program():
        host.tape_reset()
        p = table.as_input()
        loss = (p.sgather((5000,), lambda i: [gix.sindex0([i])]) * gy).ssum0()
        return loss, host.grad(loss, [p])
    loss, grads = program()
    want = float(loss.numpy()), grads[0].numpy()
    check_dot(want[0], t[ix], y)
    graph, (loss, grads) = host.capture(program)
    try:
        for replay in range(4):
            graph.launch()
            assert float(loss.numpy()) == want[0] and np.array_equal(grads[0].numpy(), want[1]), replay
            _ = float((host.concrete(y[:333 + replay]) * 2.0).ssum0().numpy())
        table.overwrite(t[::-1].copy())
        graph.launch()
        check_dot(loss.numpy(), t[::-1][ix], y)
    finally:
        graph.free()

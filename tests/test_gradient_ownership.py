"""Gradients own their memory: writing into a forward array, into another gradient or into the cotangent that was
handed in afterwards leaves a gradient as it was, whatever views lie between the product and the input.

On the device, and without one on the checker's table whose views share memory (horc_get_api_views)."""
import numpy as np
import pytest

from conftest import capi, entry, pkg

H = pkg.hostapi


@pytest.fixture(scope="module", params=[pytest.param("views", id="cpu"), pytest.param("gpu", marks=pytest.mark.gpu)])
def host(request):
    if request.param == "gpu":
        return H.Host()
    return H.Host(capi.Lib(entry.ORACLE_LIB, "horc_", api_table="get_api_views"))


RNG = np.random.default_rng(5)
A, B, C, Z = (RNG.standard_normal((6, 4)) for _ in range(4))

# view of an input of shape (6, 4), and the cotangent of the input when that of the view is w
VIEWS = {
    "none": (lambda x: x, (6, 4), lambda w: w),
    "transpose": (lambda x: x.stranspose([1, 0]), (4, 6), lambda w: w.T),
    "reshape": (lambda x: x.sreshape([3, 8]), (3, 8), lambda w: w.reshape(6, 4)),
    "reverse": (lambda x: x.sreverse(), (6, 4), lambda w: w[::-1]),
    "slice": (lambda x: x.sslice(1, 3), (3, 4), lambda w: np.concatenate([np.zeros((1, 4)), w, np.zeros((2, 4))])),
    "transposed twice": (lambda x: x.stranspose([1, 0]).sreshape([2, 2, 6]).stranspose([2, 0, 1]), (6, 2, 2), lambda w: w.reshape(6, 4)),
}


def overwritten(v, x):
    """Every array that x's memory takes the elements of: the start of a training step's write-back."""
    v.assign(v.host.concrete(x))


@pytest.mark.parametrize("name", VIEWS)
@pytest.mark.parametrize("pending", [False, True])
def test_writes_into_the_other_factor(host, name, pending):
    view, shape, back = VIEWS[name]
    w0 = np.random.default_rng(6).standard_normal(shape)
    x, w = host.param(A), host.param(w0)
    f = w * host.concrete(np.full(shape, 2.0)) if pending else w       # the factor, and its value
    wf = w0 * 2 if pending else w0
    gx, gw = host.grad((view(x) * f).ssum0(), [x, w])
    if pending:
        f.numpy()
        overwritten(f, wf * 0 + 7)
    overwritten(w, w0 * 0 - 3)
    overwritten(x, A * 0 + 5)
    assert np.array_equal(gx.numpy(), back(wf))
    base = view(host.concrete(A)).numpy()
    assert np.array_equal(gw.numpy(), base * 2 if pending else base)
    host.tape_reset()


@pytest.mark.parametrize("name", VIEWS)
def test_plain_descent_one_parameter_after_the_other(host, name):
    view, shape, back = VIEWS[name]
    w0 = np.random.default_rng(7).standard_normal(shape)
    x, w = host.param(A), host.param(w0)
    gx, gw = host.grad((view(x) * w).ssum0(), [x, w])
    w.assign(w - gw * 0.1)
    x.assign(x - gx * 0.1)
    assert np.allclose(w.numpy(), w0 - 0.1 * view(host.concrete(A)).numpy(), rtol=1e-15)
    assert np.allclose(x.numpy(), A - 0.1 * back(w0), rtol=1e-15)
    host.tape_reset()


def test_dot_products_and_inner_contractions(host):
    x, y = host.param(A), host.param(B)
    gx, gy = host.grad(x.stranspose([1, 0]).sdot0(y.stranspose([1, 0])), [x, y])
    overwritten(x, C)
    overwritten(y, Z)
    assert np.array_equal(gx.numpy(), B) and np.array_equal(gy.numpy(), A)
    host.tape_reset()


def test_gradients_of_one_pending_factor_do_not_share(host):
    x, z, a, b = (host.param(v) for v in (A, Z, B, C))
    y = a * b
    g, g2 = host.grad((x * y).ssum0() + (z * y).ssum0(), [x, z])
    want = B * C
    overwritten(g2, A)
    assert np.array_equal(g.numpy(), want)
    assert np.array_equal(y.numpy(), want)
    overwritten(y, Z)
    assert np.array_equal(g.numpy(), want) and np.array_equal(g2.numpy(), A)
    host.tape_reset()


def test_one_cotangent_for_two_inputs(host):
    """x + y hands one cotangent on to both."""
    x, y, w = host.param(A), host.param(B), host.concrete(C)
    gx, gy = host.grad(((x + y) * w).ssum0(), [x, y])
    overwritten(gy, Z)
    assert np.array_equal(gx.numpy(), C) and np.array_equal(gy.numpy(), Z) and np.array_equal(w.numpy(), C)
    for view in (lambda v: v, lambda v: v.stranspose([1, 0]).stranspose([1, 0]), lambda v: v.sreverse().sreverse()):
        t = x + view(y)
        gx, gy = host.grad((t * t).ssum0(), [x, y])
        overwritten(gx, Z)
        assert np.allclose(gy.numpy(), 2 * (A + B), rtol=1e-15)
        gx, gy = host.grad((t * t).ssum0(), [x, y])
        overwritten(gy, Z)
        assert np.allclose(gx.numpy(), 2 * (A + B), rtol=1e-15)
    host.tape_reset()


def test_scalars_and_the_seed(host):
    """The cotangent of an objective that is its own input is the seed: nobody can write into the library's one."""
    s = host.param(np.float64(3.0))
    g, = host.grad(s * host.concrete(np.float64(2.0)), [s])
    g, = host.grad(s.sreshape([]), [s])
    assert g.numpy() == 1.0
    overwritten(g, np.float64(9.0))
    h, = host.grad(s.sreshape([]), [s])
    assert h.numpy() == 1.0 and g.numpy() == 9.0
    # nor into its zero
    u, v = host.param(np.float64(1.0)), host.param(np.float64(2.0))
    for _ in range(2):
        gu, gv, gs = host.grad(s * s, [u, v, s])
        assert gu.numpy() == 0.0 and gv.numpy() == 0.0 and gs.numpy() == 6.0
        overwritten(gu, np.float64(9.0))
        assert gv.numpy() == 0.0
    # a cotangent that the caller brings is the caller's array
    x, dt = host.param(A), host.concrete(B)
    g, = host.grad(x.sreshape([6, 4]), [x], dt=dt)
    overwritten(dt, C)
    assert np.array_equal(g.numpy(), B)
    host.tape_reset()


@pytest.mark.parametrize("name", ["transpose", "reverse", "sum", "rows' sums"])
def test_strided_views_of_the_callers_cotangent(host, name):
    """Views that cannot be written into themselves change with the array behind them all the same."""
    ops = {"transpose": (lambda x: x.stranspose([1, 0]), lambda d: d.T), "reverse": (lambda x: x.sreverse(), lambda d: d[::-1]),
           "sum": (lambda x: x.ssum0(), lambda d: np.broadcast_to(d, (6, 4))),
           "rows' sums": (lambda x: x.stranspose([1, 0]).ssum(), lambda d: np.broadcast_to(d[:, None], (6, 4)))}
    op, back = ops[name]
    x = host.param(A)
    out = op(x)
    d = np.random.default_rng(9).standard_normal(out.shape)
    dt = host.concrete(d)
    g, = host.grad(out, [x], dt=dt)
    overwritten(dt, d * 0 + 7)
    assert np.array_equal(g.numpy(), back(d))
    host.tape_reset()


@pytest.mark.parametrize("swap", [False, True])
@pytest.mark.parametrize("name", ["transpose", "reverse", "sum", "rows' sums"])
def test_writes_into_a_gradient_that_another_one_is_a_view_of(host, name, swap):
    y0 = {"transpose": B.T, "reverse": B, "sum": np.float64(2.0), "rows' sums": B[:, 0]}[name]
    op = {"transpose": lambda x: x.stranspose([1, 0]), "reverse": lambda x: x.sreverse(), "sum": lambda x: x.ssum0(),
          "rows' sums": lambda x: x.stranspose([1, 0]).ssum()}[name]
    x, y = host.param(A), host.param(y0)
    t = op(x) + y
    inputs = [y, x] if swap else [x, y]

    def gradients():
        gs = host.grad((t * t).ssum0() if t.shape else t * t, inputs)
        return gs[::-1] if swap else gs
    gx, gy = gradients()
    want = gx.numpy().copy()
    wanty = gy.numpy().copy()
    overwritten(gy, wanty * 0 + 7)
    assert np.array_equal(gx.numpy(), want)
    gx, gy = gradients()
    try:
        overwritten(gx, want * 0 + 7)
    except capi.HgpuError:         # a view that is refused as a destination
        assert np.array_equal(gx.numpy(), want)
    assert np.array_equal(gy.numpy(), wanty)
    host.tape_reset()


def test_gradients_are_destinations(host):
    """What a gradient was taken through does not show in whether it can be written into."""
    for name, (view, shape, back) in VIEWS.items():
        x, w = host.param(A), host.param(np.ones(shape))
        gx, gw = host.grad((view(x) * w).ssum0(), [x, w])
        if name != "slice":
            overwritten(gx, Z)
            assert np.array_equal(gx.numpy(), Z), name
        overwritten(gw, np.zeros(shape))
        assert np.array_equal(w.numpy(), np.ones(shape)), name
        host.tape_reset()


def test_slices_of_one_cotangent(host):
    """Neighbouring slices of one array share a block of memory and no element: nothing is copied for them."""
    x, y, w = host.param(A), host.param(B), host.concrete(np.concatenate([C, Z]))
    t = x.sappend(y) * w
    gx, gy = host.grad((t * t).ssum0(), [x, y])
    want = 2 * np.concatenate([A * C * C, B * Z * Z])
    overwritten(gx, Z)
    assert np.allclose(gy.numpy(), want[6:], rtol=1e-14) and np.array_equal(gx.numpy(), Z)
    host.tape_reset()


@pytest.mark.gpu
def test_shares_memory(gpu):
    a = gpu.upload(np.zeros((6, 4)))
    shares = lambda x, y: gpu.lib.shares_memory(x.h, y.h)
    top, low, mid = a.slice(0, 0, 3), a.slice(0, 3, 3), a.slice(0, 2, 3)
    assert shares(a, top) and shares(a, a.transpose([1, 0])) and shares(mid, top) and shares(mid, low)
    assert not shares(top, low) and not shares(top.transpose([1, 0]), low.reverse(0)) and not shares(low.reverse(1), top.reverse(0))
    assert shares(top.reverse(0), mid.reverse(1)) and shares(a.slice(1, 0, 2), a.slice(1, 2, 2))      # (rows interleave)
    assert not shares(a, gpu.upload(np.zeros((6, 4)))) and not shares(a, a.slice(0, 2, 0))
    s = a.slice(0, 5, 1).slice(1, 3, 1).reshape([])
    assert shares(s, low) and not shares(s, top) and shares(s.replicate([7]), low) and not shares(s.replicate([7]), top)


@pytest.mark.gpu
@pytest.mark.parametrize("name", VIEWS)
def test_recorded_step_returns_gradients_of_the_old_parameters(name):
    view, shape, back = VIEWS[name]
    host = H.Host()
    w0 = np.random.default_rng(8).standard_normal(shape)
    x, w = host.param(A), host.param(w0)

    def step():
        gx, gw = host.grad((view(x) * w).ssum0(), [x, w])
        w.assign(w - gw * 0.1)
        x.assign(x - gx * 0.1)
        return gx, gw
    step()
    x.overwrite(A)
    w.overwrite(w0)
    host.sync()
    graph, (gx, gw) = host.capture(step)
    xs, ws = A.copy(), w0.copy()
    for _ in range(3):
        graph.launch()
        host.sync()
        base = view(host.concrete(xs)).numpy()
        assert np.allclose(gx.numpy(), back(ws), rtol=1e-14) and np.allclose(gw.numpy(), base, rtol=1e-14)
        xs, ws = xs - 0.1 * back(ws), ws - 0.1 * base
        assert np.allclose(x.numpy(), xs, rtol=1e-14) and np.allclose(w.numpy(), ws, rtol=1e-14)
    graph.free()


@pytest.mark.gpu
def test_recorded_program_follows_the_callers_cotangent():
    host = H.Host()
    x, w, dt = host.param(A), host.concrete(B), host.srepl((), 1.0)

    def step():
        return host.grad((x * w).ssum0(), [x], dt=dt)
    step()
    graph, (g,) = host.capture(step)
    for f in (1.0, 2.0, -0.5):
        dt.overwrite(np.float64(f))
        graph.launch()
        host.sync()
        assert np.array_equal(g.numpy(), B * f)
    graph.free()

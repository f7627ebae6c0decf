"""The reductions of a small objective as one launch (HeadJob in csrc/fused.hip): extremum, sum and map with sums over the same
elements.  Against numpy in long doubles; sums are formed in double, a few dozen roundings of the type lie between."""
import ctypes as C

import numpy as np
import pytest

from conftest import capi, pkg
import test_held_sums as held

H, W = pkg.hostapi, pkg.workloads
pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def host():
    return H.Host()


def reference(x, y):
    x, y = x.astype(np.longdouble), y.astype(np.longdouble)
    e = np.exp(x - x.min())
    soft = e / e.sum()
    return float(-(np.log(soft) * y).sum()), (soft - y).astype(np.float64)


@pytest.mark.parametrize("dt", [np.float64, np.float32])
@pytest.mark.parametrize("classes,batch", [(10, 6), (10, 7), (7, 13), (10, 204), (10, 205), (3, 683), (10, 409), (8, 512), (17, 241), (2, 4096), (3, 2731), (10, 1000)])
def test_soft_max_cross_entropy(host, dt, classes, batch):
    """From 64 elements to 32 KB, whole vectors and not, one block's single trip and several."""
    one = 64 <= classes * batch <= 32768 // np.dtype(dt).itemsize
    rng = np.random.default_rng(batch)
    x, y = rng.uniform(-2, 2, (classes, batch)).astype(dt), rng.uniform(0, 1, (classes, batch)).astype(dt)
    px, py = host.param(x), host.concrete(y)

    def program():
        host.tape_reset()
        p = px.as_input()
        loss = W.lossSoftMaxCrossEntropyS(py, p)
        return loss, host.grad(loss, [p])[0]
    eager = [v.numpy() for v in program()]
    graph, res, labels = held.recorded(host, program)
    assert sum(k.startswith("fused_head") for k in labels) == one and sum(k.startswith("argminmax") for k in labels) == (not one), labels
    want_loss, want = reference(x, y)
    eps = np.finfo(dt).eps
    try:
        for _ in range(3):
            graph.launch()
            loss, grad = [v.numpy() for v in res]
            assert np.array_equal(loss, eager[0]) and np.array_equal(grad, eager[1])
            assert abs(float(loss) - want_loss) <= 64 * eps * abs(want_loss)
            assert np.all(np.abs(grad - want) <= 16 * eps * np.maximum(np.abs(want), 1))
            [v.numpy() for v in program()]
    finally:
        graph.free()


@pytest.mark.parametrize("dt", [np.float64, np.float32])
@pytest.mark.parametrize("n", [64, 1000, 4096, 4097, 8193])
@pytest.mark.parametrize("kind", ["min", "max"])
def test_extremum_alone_and_in_a_program(host, dt, n, kind):
    """Ties, NaNs and infinities; its value read at once, by an elementwise pass, by a sum, by both."""
    rng = np.random.default_rng(n)
    base = rng.integers(-5, 6, n).astype(dt)
    for case in ("ties", "nan first", "nan inside", "all nan", "inf"):
        x = base.copy()
        if case == "nan first":
            x[0] = np.nan
        if case == "nan inside":
            x[1::3] = np.nan
        if case == "all nan":
            x[:] = np.nan
        if case == "inf":
            x[n // 2], x[n // 3] = np.inf, -np.inf
        v = host.concrete(x)
        arg = (v.sargMin if kind == "min" else v.sargMax)()
        val = v.sgather((), lambda: [arg.lift(())])
        if np.isnan(x[0]):
            at = 0
        else:
            at = int(np.nanargmin(x) if kind == "min" else np.nanargmax(x))
        shifted = (v - val.sreplicate0N([n])) * 0.25
        total = shifted.ssum0()
        with np.errstate(invalid="ignore"):
            s = (x - x[at]) * dt(0.25)
        assert np.array_equal(total.numpy(), dt(s.astype(np.float64).sum()), equal_nan=True), case
        assert np.array_equal(val.numpy(), x[at], equal_nan=True), case
        assert int(arg.numpy()) == at, case
        assert np.array_equal(shifted.numpy(), s, equal_nan=True), case


def test_what_waits_goes_out_for_its_readers(host):
    """The logits are a product that is held itself; the extremum is read between the phases; the logits are overwritten after."""
    rng = np.random.default_rng(1)
    w, x, y = rng.uniform(-1, 1, (10, 30)), rng.uniform(-1, 1, (30, 64)), rng.uniform(0, 1, (10, 64))
    pw, px, py = host.param(w), host.concrete(x), host.concrete(y)

    def program(peek):
        host.tape_reset()
        p = pw.as_input()
        d = p.smatmul2(px)
        u = d.sprimalPart()
        lo = W.sminimum(u)
        if peek == "value":
            lo.numpy()
        e = (u - lo.sreplicate0N(u.shape)).op1("exp")
        total = e.ssum0()
        if peek == "sum":
            total.numpy()
        soft = total.op1("recip").sreplicate0N(u.shape) * e
        primal = -(soft.op1("log").sdot0(py))
        loss = primal.tD((soft - py).sdot0(d))
        return loss, host.grad(loss, [p])[0]
    want_loss, cot = reference(w @ x, y)
    for peek in (None, "value", "sum"):
        loss, grad = [v.numpy() for v in program(peek)]
        assert abs(float(loss) - want_loss) <= 1e-12 * abs(want_loss), peek
        assert np.allclose(grad, cot @ x.T, rtol=1e-11, atol=1e-12), peek
    z = host.concrete(x[0].copy())
    arg = z.sargMax()
    val = z.sgather((), lambda: [arg.lift(())])
    z.overwrite(-x[0])
    assert float(val.numpy()) == x[0].max() and int(arg.numpy()) == int(x[0].argmax())

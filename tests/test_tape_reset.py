"""Values that outlive the tape they were recorded on are constants to what is recorded next (Tape::reset, host/adval.cpp): the
objective's value that Workload.gradient returns, whose tape goes when the gradients have been asked for, among them."""
import numpy as np
import pytest

from conftest import capi, entry, pkg

H = pkg.hostapi


@pytest.fixture(scope="module", params=[pytest.param("cpu", id="cpu"), pytest.param("gpu", marks=pytest.mark.gpu)])
def host(request):
    if request.param == "gpu":
        return H.Host()
    return H.Host(capi.Lib(entry.ORACLE_LIB, "horc_", api_table="get_api_views"))


A = np.arange(1.0, 7.0)


@pytest.mark.parametrize("before", [0, 1, 40])
def test_a_value_of_another_tape_is_a_constant(host, before):
    host.tape_reset()
    x = host.param(A)
    old = x
    for _ in range(before):
        old = old * 1.5
    old = old * x
    want_old = A * A * 1.5 ** before
    host.tape_reset()
    w = host.param(A + 1)
    y = host.param(A + 2)
    gw, gy = host.grad((old * w + y * y).ssum0(), [w, y])
    assert np.allclose(gw.numpy(), want_old, rtol=1e-14) and np.array_equal(gy.numpy(), 2 * (A + 2))
    (gw,) = host.grad((old * 2.0).ssum0(), [w])
    assert np.array_equal(gw.numpy(), 0 * A)
    host.tape_reset()


def test_the_value_of_a_gradient_goes_into_the_next_program(host):
    wl = pkg.workloads.Workload("square", np.float64, 1, [A], [], lambda ps, ds: (ps[0] * ps[0]).ssum0(), 1, 1)
    ps, ds = wl.upload(host)
    loss, (g,) = wl.gradient(host, ps, ds)
    w = host.param(A)
    (gw,) = host.grad((loss.sreplicate0N([6]) * w).ssum0() if hasattr(loss, "sreplicate0N") else (w * loss).ssum0(), [w])
    assert np.array_equal(g.numpy(), 2 * A) and np.array_equal(gw.numpy(), np.full(6, (A * A).sum()))
    (gw,) = host.grad(loss, [w])
    assert np.array_equal(gw.numpy(), 0 * A)
    host.tape_reset()


def test_the_derivative_by_an_input_of_another_tape_is_refused(host):
    x = host.param(A)
    host.tape_reset()
    y = x.as_input()
    with pytest.raises(Exception, match="reset"):
        host.grad((x * y).ssum0(), [x])
    (gy,) = host.grad((x * y).ssum0(), [y])
    assert np.array_equal(gy.numpy(), A)
    host.tape_reset()

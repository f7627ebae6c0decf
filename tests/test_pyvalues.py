"""Values and calls of the CPython extension (host/pyvalues.cpp), on the CPU checker."""
import gc
import os
import subprocess
import sys
import sysconfig
import threading
import weakref

import numpy as np
import pytest

from conftest import capi, entry, pkg

H = pkg.hostapi


@pytest.fixture(scope="module")
def host():
    return H.Host(api_lib=capi.Lib(entry.ORACLE_LIB, "horc_"))


def test_integers_as_python_has_them(host):
    """Shapes, permutations and indices from lists, tuples, ranges and numpy, empty ones included."""
    x = np.arange(24.0).reshape(2, 3, 4)
    v = host.concrete(x)
    for perm in ([2, 0, 1], (2, 0, 1), np.array([2, 0, 1], np.int32)):
        assert np.array_equal(v.stranspose(perm).numpy(), x.transpose(2, 0, 1))
    for shape in ([6, 4], (np.int64(6), 4), range(24, 25)):
        assert np.array_equal(v.sreshape(shape).numpy(), x.reshape(tuple(int(s) for s in shape)))
    assert np.array_equal(v.sindex([1, np.int64(2)]).numpy(), x[1, 2]) and np.array_equal(v.sindex([]).numpy(), x)
    assert v.sreplicateN([]).shape == (2, 3, 4) and v.sreplicate(np.int32(5)).shape == (5, 2, 3, 4)
    assert np.array_equal(v.sslice(True, 1).numpy(), x[1:2])
    assert host.srepl((), 3).numpy() == 3.0 and host.srepl((2,), np.float32(0.5), capi.F32).numpy().tolist() == [0.5, 0.5]
    assert host.siota(n=3).numpy().tolist() == [0, 1, 2] and v.sslice(i=0, n=2).shape == (2, 3, 4) and v.sdotNIn(v, n=2).shape == (2,)


@pytest.mark.parametrize("wrong", [
    lambda h, v: v.sslice(1.7, 2.2), lambda h, v: v.sslice("1", "2"), lambda h, v: v.sslice(0, np.float64(2)), lambda h, v: v.ssumN(1.9), lambda h, v: h.siota(3.9),
    lambda h, v: h.siota("3"), lambda h, v: v.stranspose([1.0, 0.9, 2]), lambda h, v: v.stranspose("102"), lambda h, v: v.stranspose([2 ** 32 + 1, 0, 2]),
    lambda h, v: v.ssumN(2 ** 32 + 1), lambda h, v: v.ssumN(1 - 2 ** 32), lambda h, v: v.sslice(2 ** 64, 2), lambda h, v: v.sdotNIn(v, 1.5), lambda h, v: v.scast(2 ** 33)])
def test_no_integers(host, wrong):
    """Fractions, texts and what the parameter cannot hold are refused, not cut to an integer."""
    with pytest.raises((TypeError, OverflowError)):
        wrong(host, host.concrete(np.arange(24.0).reshape(2, 3, 4)))


def test_sizes_are_what_int_gives(host):
    v = host.concrete(np.arange(24.0))
    assert v.sreshape([6.0, 4]).shape == v.sreshape(["6", np.float32(4)]).shape == (6, 4) and v.sreplicate(2.5).shape == (2, 24)
    assert v.sslice(np.int64(5), np.int8(2)).numpy().tolist() == [5, 6] and host.siota(2 ** 33 % 7).shape == (2 ** 33 % 7,)
    with pytest.raises(OverflowError):
        v.sreshape([2 ** 64, 1])


def test_lane_values(host):
    v = host.concrete(np.arange(12.0).reshape(3, 4))
    seen = []

    def f(i, j):
        seen.extend([i, j, i + 1, 2 - j, i * j, -i])
        return [j - 1, 2 - i]
    got = v.sgather((3, 4), f).numpy()
    x = np.arange(12.0).reshape(3, 4)
    want = np.array([[x[j - 1, 2 - i] if 0 <= j - 1 < 3 and 0 <= 2 - i < 4 else 0 for j in range(4)] for i in range(3)])
    assert np.array_equal(got, want)
    assert all(s.shm == (3, 4) and s.host is host for s in seen) and seen[0].dtype == capi.I64 and seen[0].is_affine
    assert H.IxV.from_val(v).shm == (3, 4) and H.IxV.from_val(v).dtype == capi.F64
    assert v.sgather((), lambda: [1, 2]).numpy() == x[1, 2]


def test_errors(host):
    v = host.concrete(np.zeros((2, 3)))
    with pytest.raises(H.HgpuError) as e:
        v.sreshape([7])
    assert e.value.code != 0 and "status" in str(e.value)
    with pytest.raises(H.HgpuError):
        v.smatmul2(v)
    for wrong in (lambda: v.smatmul2(3), lambda: v.sreshape(5), lambda: v.sreshape(["a"]), lambda: v.sappend(None), lambda: v.sgather((2,), lambda i: [v]),
                  lambda: v.op2("add", "x"), lambda: host.grad(v, [3])):
        with pytest.raises((TypeError, ValueError, AttributeError)):
            wrong()
    with pytest.raises(KeyError):
        v.op1("no such operation")
    with pytest.raises(ValueError):
        v.sreplicateN([1] * 100)


def test_values_go_when_nobody_has_them(host):
    v = host.concrete(np.ones(4))
    assert isinstance(v.h, int) and v.host is host
    w = weakref.ref(v)
    v.note = [v]                       # a cycle through the value's own attributes
    del v
    gc.collect()
    assert w() is None
    again = host.concrete(np.arange(3.0))
    kept = [again * k for k in range(200)]
    del kept
    assert np.array_equal(again.numpy(), np.arange(3.0))


def test_built_from_the_source_that_is_there(tmp_path):
    source = os.path.join(capi.HERE, "host", "pyvalues.cpp")
    H._check_source(H._py.SOURCE, source)
    H._check_source(H._py.SOURCE, str(tmp_path / "none"))
    changed = tmp_path / "pyvalues.cpp"
    with open(source) as f:
        changed.write_text(f.read() + "// another line\n")
    with pytest.raises(ImportError, match="build"):
        H._check_source(H._py.SOURCE, str(changed))
    assert H.EXTENSION.endswith(sysconfig.get_config_var("EXT_SUFFIX")) and os.path.samefile(H._py.__file__, H.EXTENSION)


ITERATORS = """
import numpy as np
from conftest import capi, entry, pkg
H = pkg.hostapi
host = H.Host(api_lib=capi.Lib(entry.ORACLE_LIB, "horc_"))
x = np.arange(12.0).reshape(3, 4)
v = host.concrete(x)
for _ in range(300):
    got = H._c.tsgather(host, v, (3, 4), ((i + 0 for i in host.ix_space((3, 4)))))
    assert np.array_equal(got.numpy(), x)
    lane = H._c.ix_index0(host, v, (i + 0 for i in host.ix_space((3, 4))))
    assert lane.shm == (3, 4) and np.array_equal(lane.to_val().numpy(), x)
    p = v.as_input()
    host.tape_reset()
    loss = (p * p).ssum0()
    assert [g.shape for g in host.grad(loss, (v * k for k in (1.0, 2.0)))] == [(3, 4)] * 2
print("all of them")
"""


def test_arguments_that_nobody_else_has():
    """Lane values and inputs that an iterator makes live until the call is over (in a process of its own: what reads freed memory may end it)."""
    r = subprocess.run([sys.executable, "-c", ITERATORS], cwd=os.path.dirname(os.path.abspath(__file__)), stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True, timeout=100)
    assert r.returncode == 0 and "all of them" in r.stdout, r.stdout[-2000:]


def test_threads_with_contexts_of_their_own():
    errors = []

    def work(k):
        try:
            h = H.Host(api_lib=capi.Lib(entry.ORACLE_LIB, "horc_"))
            x = h.param(np.full(64, float(k)))
            for _ in range(50):
                h.tape_reset()
                p = x.as_input()
                loss = (p * p).ssum0()
                g, = h.grad(loss, [p])
                assert float(loss.numpy()) == 64 * k * k and np.array_equal(g.numpy(), np.full(64, 2.0 * k))
        except Exception as e:      # noqa: BLE001
            errors.append(e)
    ts = [threading.Thread(target=work, args=(k,)) for k in range(4)]
    [t.start() for t in ts]
    [t.join() for t in ts]
    assert not errors, errors

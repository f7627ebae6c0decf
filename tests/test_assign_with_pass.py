"""Copies into existing arrays that wait with the elementwise pass whose result they take (copy_with_map_locked, csrc/smallk.hip):
inside a recording the pass writes to their destination, where nobody else has its result."""
import ctypes as C

import numpy as np
import pytest

import test_held_sums as held
from conftest import pkg

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def host():
    return pkg.hostapi.Host()


def update(host, s, keep):
    """An optimizer's: every new value from the old ones."""
    a, b, c, d = s
    m = a * 0.5 + d * 0.25
    v = b * 0.75 + d * d
    p = c - m * v
    host.submit(m, v, p)
    for dst, src in ((a, m), (b, v), (c, p)):
        dst.assign(src)
    return []


def swap(host, s, keep):
    a, b, c, d = s
    x, y = b * 2.0, a * 3.0
    host.submit(x, y)
    a.assign(x)
    b.assign(y)
    return []


def kept(host, s, keep):
    a, b, c, d = s
    x = a * b + c
    host.submit(x)
    a.assign(x)
    return [x, x * 2.0]


def kept_outside(host, s, keep):
    a, b, c, d = s
    x = a * b + c
    host.submit(x)
    a.assign(x)
    keep.append(x)
    return []


def twice(host, s, keep):
    a, b, c, d = s
    x, y = a + c * 0.5, b - a * 0.5
    host.submit(x, y)
    a.assign(x)
    b.assign(x)          # the same result to two places
    c.assign(y)
    c.assign(d)          # ... and two results to one
    return []


def read_after(host, s, keep):
    a, b, c, d = s
    x = a * 0.5 + b
    host.submit(x)
    a.assign(x)
    y = a * 2.0          # reads what the pass has written
    b.assign(y)
    return [a + b]


def another_input(host, s, keep):
    """The destination is an input of the pass that the result does not come from."""
    a, b, c, d = s
    x, y = b + c, a * 2.0 - b
    host.submit(x, y)
    a.assign(x)
    d.assign(y)
    return []


PROGRAMS = {
    update: lambda a, b, c, d: (a * 0.5 + d * 0.25, b * 0.75 + d * d, c - (a * 0.5 + d * 0.25) * (b * 0.75 + d * d), d),
    swap: lambda a, b, c, d: (b * 2, a * 3, c, d),
    kept: lambda a, b, c, d: (a * b + c, b, c, d),
    kept_outside: lambda a, b, c, d: (a * b + c, b, c, d),
    twice: lambda a, b, c, d: (a + c * 0.5, a + c * 0.5, d, d),
    read_after: lambda a, b, c, d: (a * 0.5 + b, (a * 0.5 + b) * 2, c, d),
    another_input: lambda a, b, c, d: (b + c, b, c, a * 2 - b),
}


@pytest.mark.parametrize("shape", [(1,), (), (3,), (4, 1), (127, 65), (1024, 257)])
@pytest.mark.parametrize("program", list(PROGRAMS), ids=lambda f: f.__name__)
@pytest.mark.parametrize("dt", [np.float64, np.float32])
def test_recorded_updates(host, program, shape, dt):
    rng = np.random.default_rng(len(shape) + 1)
    x = [rng.uniform(-1, 1, shape).astype(dt) for _ in range(4)]
    s = [host.concrete(v) for v in x]
    keep = []
    program(host, s, keep)                       # the program's constants
    for v, a in zip(x, s):
        a.overwrite(v)
    graph, res, labels = held.recorded(host, lambda: program(host, s, keep))
    if program is update:
        assert "copy_group" not in labels, labels
    cur = [v.astype(np.float64) for v in x]
    eps = np.finfo(dt).eps
    try:
        for step in range(4):
            graph.launch()
            host.sync()
            old, cur = cur, [np.asarray(v, np.float64) for v in PROGRAMS[program](*cur)]
            bound = 64 * eps * (1 + sum(np.abs(v) for v in old)) ** 2 * 3 ** step
            got = [a.numpy() for a in s]
            for g, w in zip(got, cur):
                assert np.all(np.abs(g - w) <= bound), (program.__name__, step)
            for r, w in zip(res, {kept: [cur[0], cur[0] * 2], read_after: [cur[0] + cur[1]]}.get(program, [])):
                assert np.all(np.abs(r.numpy() - w) <= 4 * bound)
            if program is kept_outside:
                assert np.array_equal(keep[-1].numpy(), got[0])
            cur = [g.astype(np.float64) for g in got]
    finally:
        graph.free()


def test_destinations_amid_an_array(gpu):
    """A part of an array that does not start on 16 bytes, beside the same part on 16 bytes."""
    dll = gpu.lib.dll
    rng = np.random.default_rng(5)
    x, y = rng.uniform(-1, 1, (2, 300))
    a, b, whole = gpu.upload(x), gpu.upload(y), gpu.upload(np.zeros(1000))
    prog = [(1, pkg.capi.OP2["add"], 0, 0, 1, 0)]
    gpu.fused_map([a, b], prog, [2])
    gpu.check(dll.hgpu_capture_begin(gpu.h))
    for first in (1, 302, 604):
        part = whole.slice(0, first, 300)
        part.assign(gpu.fused_map([a, b], prog, [2])[0])
    g = C.c_void_p()
    gpu.check(dll.hgpu_capture_end(gpu.h, C.byref(g)))
    try:
        for _ in range(3):
            gpu.check(dll.hgpu_graph_launch(g))
            want = np.zeros(1000)
            for first in (1, 302, 604):
                want[first:first + 300] = x + y
            assert np.array_equal(whole.numpy(), want)
            whole.assign(gpu.upload(np.zeros(1000)))
    finally:
        gpu.check(dll.hgpu_graph_destroy(g))


@pytest.mark.parametrize("dt", [np.float64, np.float32])
def test_two_results_of_an_input_that_one_is_written_to(dt, tmp_path, monkeypatch):
    """The other result reads the overwritten input too: the kernel promises the compiler nothing about which arrays are apart, and
    every replay gives the bits of the pass into new arrays."""
    monkeypatch.setenv("HORDEAD_GPU_KEEP_SOURCES", str(tmp_path))
    ctx = pkg.capi.Lib().context(0)                  # (none of its kernels is known yet)
    dll, O2 = ctx.lib.dll, pkg.capi.OP2
    prog = [(1, O2["mul"], 0, 0, 1, 0), (1, O2["add"], 0, 2, 0, 0), (1, O2["sub"], 0, 0, 3, 0)]
    rng = np.random.default_rng(7)
    x, y = rng.uniform(-1, 1, (2, 70003)).astype(dt)
    a, b, c = ctx.upload(x), ctx.upload(y), ctx.upload(np.zeros_like(x))
    want = []
    now = ctx.upload(x)
    for _ in range(3):
        now, other = ctx.fused_map([now, b], prog, [3, 4])
        want.append((now.numpy(), other.numpy()))
    ctx.profile(2)
    g = C.c_void_p()
    ctx.check(dll.hgpu_capture_begin(ctx.h))
    r = ctx.fused_map([a, b], prog, [3, 4])
    a.assign(r[0])
    c.assign(r[1])
    del r
    ctx.check(dll.hgpu_capture_end(ctx.h, C.byref(g)))
    assert not any("copy" in n for n in ctx.profile_report())
    ctx.profile(0)
    try:
        for wa, wc in want:
            ctx.check(dll.hgpu_graph_launch(g))
            assert np.array_equal(a.numpy(), wa) and np.array_equal(c.numpy(), wc)
    finally:
        ctx.check(dll.hgpu_graph_destroy(g))
    texts = [t for t in (f.read_text() for f in tmp_path.iterdir()) if "fused_map_group(" in t]
    assert len(texts) == 1 and "__restrict__" not in texts[0]

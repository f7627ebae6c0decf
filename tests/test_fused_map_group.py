"""Small elementwise passes of one kernel that a recording holds go out together (csrc/smallk.hip, launch_maps)."""
import numpy as np
import pytest

from conftest import pkg

pytestmark = pytest.mark.gpu
OPT = pkg.optimizer


@pytest.fixture(scope="module")
def host():
    return pkg.hostapi.Host()


@pytest.mark.parametrize("dt", [np.float64, np.float32])
def test_updates_of_parameters_of_many_sizes(host, dt):
    """More passes than one launch takes, with sizes around vectors and blocks, and one that goes alone."""
    rng = np.random.default_rng(1)
    sizes = [2, 3, 5, 255, 256, 257, 511, 512, 513, 1023, 1025, 4099, 70001, 2, 3, 17, 100352, 16, 25, 400, 1280, 10, 7, (1 << 20) + 1]
    p0, g0 = ([rng.uniform(-1, 1, n).astype(dt) for n in sizes] for _ in range(2))
    ps, gs = [host.concrete(p) for p in p0], [host.concrete(g) for g in g0]
    ms, vs = ([host.concrete(np.zeros(n, dt)) for n in sizes] for _ in range(2))
    args = OPT.ArgsAdam(alpha=0.01)
    alphat = host.concrete(np.asarray(0.01, dt))

    def step():
        new = OPT.adamApply(args, alphat, ms, vs, ps, gs)
        for dst, src in zip(ms + vs + ps, new[0] + new[1] + new[2]):
            dst.assign(src)
        return ps

    step()                                   # kernels and constants
    for x, was in zip(ms + vs + ps, [np.zeros(n, dt) for n in sizes * 2] + p0):
        x.overwrite(was)
    graph, _ = host.capture(step)
    try:
        for _ in range(3):
            graph.launch()
        host.sync()
        for n, p, p1, g in zip(sizes, ps, p0, g0):
            m, v, q, g = np.zeros(n), np.zeros(n), p1.astype(np.float64), g.astype(np.float64)
            for _ in range(3):
                m, v = 0.9 * m + (1 - 0.9) * g, 0.999 * v + (1 - 0.999) * g * g
                q = q - 0.01 * m / (np.sqrt(v) + args.epsilon)
            # steps of at most 0.01 * m / sqrt(v) <= 0.1 each, some ten roundings and the constants' own
            assert np.max(np.abs(p.numpy() - q)) <= 3 * (1 + 0.1 * 16) * np.finfo(dt).eps * 8, n
    finally:
        graph.free()


def test_passes_that_read_one_anothers_results_and_memory_that_is_written_again(host):
    rng = np.random.default_rng(2)
    x = [rng.uniform(0.2, 0.8, n) for n in (300, 300, 500)]
    a, b, c = (host.concrete(v) for v in x)

    def now(v):
        host.check(host.dll.hh_force(host.h, v.h))
        return v

    def program():
        s = now((a + b) * b)
        u = now((c + c) * c)               # independent: together with s
        t = now((s + b) * b)               # reads a held result
        a.assign(t)                        # written after it was read
        v = now((a + s) * s)
        return s, u, t, v

    program()
    a.overwrite(x[0])
    graph, res = host.capture(program)
    try:
        want_a = x[0]
        for _ in range(3):
            graph.launch()
            host.sync()
            s = (want_a + x[1]) * x[1]
            t = (s + x[1]) * x[1]
            for got, want in zip(res, (s, 2 * x[2] * x[2], t, (t + s) * s)):
                np.testing.assert_allclose(got.numpy(), want, rtol=4e-16 * 8, atol=0)
            want_a = t
    finally:
        graph.free()

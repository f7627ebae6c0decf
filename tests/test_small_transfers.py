"""Bytes that go to the device with a launch's arguments and come back through pinned memory (GPU only).

Sizes lie on both sides of the limits (256 bytes to the device, 4096 back) and of a wavefront's share;
a slice at an odd offset takes the units its alignment allows."""
import numpy as np
import pytest

from conftest import capi, pkg

H = pkg.hostapi
pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [np.int8, np.float32, np.float64])
@pytest.mark.parametrize("nbytes", [8, 16, 248, 256, 264, 1024, 1032, 4088, 4096, 4104])
def test_round_trip(gpu, dtype, nbytes):
    n = nbytes // np.dtype(dtype).itemsize
    rng = np.random.default_rng(nbytes)
    x = rng.integers(-100, 100, n).astype(dtype)
    mine = x.copy()
    a = gpu.upload(mine)
    mine[:] = 0                                   # the caller's memory is the caller's again
    assert np.array_equal(a.numpy(), x)
    for lo in (1, 3):                             # neither 16- nor, in bytes, 4-aligned
        if n > lo:
            assert np.array_equal(a.slice(0, lo, n - lo).numpy(), x[lo:])
    odd = gpu.upload(x[:max(n - 1, 1)])
    assert np.array_equal(odd.numpy(), x[:max(n - 1, 1)])
    assert np.array_equal(a.numpy(), x)           # the staging memory is not the array's


def test_overwrite_is_in_order_and_takes_a_copy():
    host = H.Host()
    v = host.concrete(np.zeros(5))
    graph, out = host.capture(lambda: v * v + v)
    try:
        x = np.empty(5)
        outs = []
        for k in range(40):                       # nothing waits between an overwrite and the launch that reads it
            x[:] = np.arange(5) + k
            v.overwrite(x)
            graph.launch()
            x[:] = np.nan
            outs.append(out.numpy())
        for k, o in enumerate(outs):
            w = np.arange(5.0) + k
            assert np.array_equal(o, w * w + w)
    finally:
        graph.free()


@pytest.mark.parametrize("kernels", [1, 2, 4, 5])
def test_short_recordings_replay(kernels):
    """Recordings of up to four kernels are launched one by one, longer ones as a graph: each replay reads its inputs
    anew and gives the bits of the eager run, with eager work between the replays.  Column sums of ever narrower
    arrays: run-time compiled and precompiled kernels in one chain."""
    host = H.Host()
    rng = np.random.default_rng(kernels)
    x = rng.uniform(-1, 1, (3,) * kernels + (2000,))
    v = host.concrete(x)

    def program():
        y = v
        for k in range(kernels):
            y = y.op1("sin") if k % 2 == 0 else y.ssum()
            y = y.dense()
        return y
    want = program().numpy()
    graph, out = host.capture(program)
    try:
        for replay in range(4):
            graph.launch()
            assert np.array_equal(out.numpy(), want), replay
            _ = (host.concrete(rng.uniform(-1, 1, 333 + replay)) * 2.0).numpy()
            graph.launch()
            graph.launch()
            host.sync()
            assert np.array_equal(out.numpy(), want), replay
        v.overwrite(x * 0.5)
        graph.launch()
        half = out.numpy()
        assert np.array_equal(half, program().numpy()) and not np.array_equal(half, want)
    finally:
        graph.free()

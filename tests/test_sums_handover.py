"""Sums over arrays of any size are finished by the block that ends last (csrc/fused.hip, kHandOver)."""
import numpy as np
import pytest

from conftest import capi

pytestmark = pytest.mark.gpu

O1, O2 = capi.OP1, capi.OP2


@pytest.mark.parametrize("dt", [np.float64, np.float32, np.int64])
@pytest.mark.parametrize("n", [2049, 131073, 256 * 1001 + 3, 2048 * 512 + 1, 5000011])
def test_every_pass_gives_the_same_sums(gpu, dt, n):
    """From a few blocks to the largest grids, again and again into reused memory, against numpy and bit for bit."""
    rng = np.random.default_rng(n)
    x, y = ((rng.integers(-1000, 1000, n) if dt == np.int64 else rng.uniform(-1, 1, n)).astype(dt) for _ in range(2))
    a, b = gpu.upload(x), gpu.upload(y)
    wide = np.int64 if dt == np.int64 else np.float64
    prod = (x * y).astype(wide)
    want = (prod.sum(), (x + y).astype(wide).sum())
    # the sums run in 64 bits: n roundings of partial sums at most, and one to the result's type
    mag = (np.abs(prod).sum(), np.abs(x + y).astype(wide).sum())
    prog = [(1, O2["mul"], 0, 0, 1, 0), (1, O2["add"], 0, 0, 1, 0)]
    if dt == np.int64:
        prog = [(k, o, capi.I64, p, q, c) for k, o, _, p, q, c in prog]
    first = None
    for _ in range(6):
        got = [gpu.fused_sum([a, b], prog, 2).numpy(), gpu.fused_sum([a, b], prog, 3).numpy()]
        first = first or got
        for g, f, w, m in zip(got, first, want, mag):
            assert g == f
            assert abs(float(g) - float(w)) <= (0 if dt == np.int64 else n * 2.0 ** -53 * float(m) + np.finfo(dt).eps * abs(float(w)))

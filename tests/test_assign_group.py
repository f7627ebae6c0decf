"""hgpu_assign: dense copies are held back and go out together (csrc/ewise.hip, k_copy_group)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def values(rng, n, dt):
    return rng.integers(0, 2, n).astype(dt) if dt == np.bool_ else rng.integers(-100, 100, n).astype(dt)


@pytest.mark.parametrize("dt", [np.float64, np.float32, np.int16, np.int8])
def test_many_sizes_and_alignments(gpu, dt):
    """Pieces of 8192 bytes, the last 16-byte unit, arrays that start anywhere in their buffer, and more copies than one launch takes."""
    rng = np.random.default_rng(7)
    es = np.dtype(dt).itemsize
    jobs = []
    for n in [1, 2, 3, 15, 16, 17, 255, 8192 // es - 1, 8192 // es, 8192 // es + 1, 3 * 8192 // es + 5, 100003]:
        for so in (0, 1, 3):
            for do in (0, 1, 2):
                if n > 50000 and so + do > 1:
                    continue
                src, old = values(rng, n + 4, dt), values(rng, n + 4, dt)
                jobs.append((gpu.upload(src), gpu.upload(old), src, old, so, do, n))
    for s, d, _, _, so, do, n in jobs:
        d.slice(0, do, n).assign(s.slice(0, so, n))
    for s, d, src, old, so, do, n in jobs:
        want = old.copy()
        want[do:do + n] = src[so:so + n]
        assert np.array_equal(d.numpy(), want), (n, so, do)
        assert np.array_equal(s.numpy(), src)


def test_copies_that_touch_the_same_memory_keep_their_order(gpu):
    rng = np.random.default_rng(8)
    x = [rng.standard_normal(5000) for _ in range(4)]
    a, b, c, d = (gpu.upload(v) for v in x)
    b.assign(a)                                  # read after write: c gets the old a
    c.assign(b)
    a.assign(d)                                  # write after read
    d.assign(c)
    b.slice(0, 10, 20).assign(a.slice(0, 0, 20))      # write after write, two parts of one array
    b.slice(0, 30, 20).assign(a.slice(0, 7, 20))
    want_b = x[0].copy()
    want_b[10:30], want_b[30:50] = x[3][:20], x[3][7:27]
    for got, want in ((a, x[3]), (b, want_b), (c, x[0]), (d, x[0])):
        assert np.array_equal(got.numpy(), want)


def test_copies_between_other_operations(gpu):
    """Held-back copies and held-back products: each sees what was issued before it."""
    rng = np.random.default_rng(9)
    x, y, w = rng.standard_normal((64, 128)), rng.standard_normal((64, 128)), rng.standard_normal((300, 128))
    a, s = gpu.upload(x), gpu.upload(y)
    m = gpu.upload(w).replicate([64]).transpose([1, 0, 2])

    def product():
        return m.contract(a.replicate([300]), 2)

    before = product()
    a.assign(s)
    after = product()
    a.assign(gpu.upload(x).ewise2("add", s))     # the source is freed while the copy waits
    third, scaled = product(), a.ewise2("add", a)
    for got, want in ((before, w @ x.T), (after, w @ y.T), (third, w @ (x + y).T), (scaled, 2 * (x + y))):
        np.testing.assert_allclose(got.numpy(), want, rtol=0, atol=1e-12 * 128)

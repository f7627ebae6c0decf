"""The scatter-add that counts the hits of every cell (csrc/index.hip): bit-equal to the checker while no cell is hit
more than 256 times (positions of a cell are added in ascending order), within rounding of the sum of magnitudes beyond."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def check(both, src, idx, cells):
    arr, ix = both.upload(src), [both.upload(idx)]
    gpu = both.ctxs[0]
    gpu.profile(1)
    res = both.scatter_add(arr, ix, 1, [cells])
    labels = list(gpu.profile_report())
    gpu.profile(0)
    assert "scatter_counted" in labels, labels
    g, o = res.numpy()
    inside = (idx >= 0) & (idx < cells)
    hits = np.bincount(idx[inside], minlength=cells)
    short = hits <= 256
    assert np.array_equal(g[short], o[short])
    if src.dtype.kind == "f" and not short.all():
        mass = np.zeros((cells,) + src.shape[1:])
        np.add.at(mass, idx[inside], np.abs(src[inside]).astype(np.float64))
        eps = np.finfo(src.dtype).eps
        bound = (256 + hits / 256.0 + 2)[(slice(None),) + (None,) * (src.ndim - 1)] * eps * mass
        # (the checker adds a whole run front to back: its own error is hits * eps)
        assert np.all(np.abs(g - o.astype(np.float64)) <= bound + hits.reshape((-1,) + (1,) * (src.ndim - 1)) * eps * mass)
    else:
        assert np.array_equal(g, o)
    assert np.array_equal(g, both.scatter_add(arr, ix, 1, [cells]).numpy()[0])     # the same again


@pytest.mark.parametrize("dt", [np.float64, np.float32, np.int64, np.int16, np.int8])
@pytest.mark.parametrize("width", [1, 2, 7, 16, 128, 300])
def test_runs_at_the_edges_of_the_kernels(both, dt, width):
    """Cells hit 0, 1, 63 .. 65, 255 .. 257 times: a group's LDS list, a segment, one more."""
    rng = np.random.default_rng(width)
    counts = np.array([0, 1, 2, 8, 63, 64, 65, 127, 128, 129, 255, 256, 257, 0, 512, 513, 3])
    idx = rng.permutation(np.concatenate([np.repeat(np.arange(len(counts)), counts), [-1, len(counts), 1 << 40]])).astype(np.int64)
    shape = (len(idx),) if width == 1 else (len(idx), width)
    src = rng.integers(-100, 100, shape).astype(dt) if np.dtype(dt).kind == "i" else rng.standard_normal(shape).astype(dt)
    check(both, src, idx, len(counts))


@pytest.mark.parametrize("width", [1, 5])
def test_runs_longer_than_the_lds_list(both, width):
    rng = np.random.default_rng(9)
    idx = rng.permutation(np.concatenate([np.full(8192, 3), np.full(8193, 7), np.full(21001, 90), rng.integers(0, 400, 5000)])).astype(np.int64)
    src = rng.standard_normal((len(idx),) if width == 1 else (len(idx), width))
    check(both, src, idx, 400)


def test_many_cells_and_two_index_dims(both):
    rng = np.random.default_rng(10)
    i, j = rng.integers(-1, 151, 40000).astype(np.int64), rng.integers(0, 90, 40000).astype(np.int64)
    src = both.upload(rng.standard_normal((40000, 12)).astype(np.float32))
    g, o = both.scatter_add(src, [both.upload(i), both.upload(j)], 1, [150, 90]).numpy()
    assert np.array_equal(g, o)
    check(both, rng.standard_normal((3000, 32)), rng.integers(0, 25000, 3000).astype(np.int64), 25000)
    # a strided view of the data: slices that are not contiguous
    wide = both.upload(rng.standard_normal((24, 3000)))
    idx = both.upload(rng.integers(0, 700, 3000).astype(np.int64))
    g, o = both.scatter_add(wide.transpose([1, 0]), [idx], 1, [700]).numpy()
    assert np.array_equal(g, o)


def in_segments(src, idx, cells):
    """The sums in the documented order, with the type's own rounding: positions ascending, a run cut into segments of
    256 entries that are added front to back, their sums added in ascending order."""
    out = np.zeros((cells,) + src.shape[1:], src.dtype)
    order = np.argsort(idx, kind="stable")
    starts = np.searchsorted(idx[order], np.arange(cells + 1))
    for c in range(cells):
        rows = src[order[starts[c]:starts[c + 1]]]
        sums = [np.add.accumulate(rows[i:i + 256], axis=0, dtype=src.dtype)[-1] for i in range(0, len(rows), 256)]
        if sums:
            out[c] = np.add.accumulate(np.stack(sums), axis=0, dtype=src.dtype)[-1]
    return out


def counted(gpu, src, idx, cells):
    """The result and, the same again, the kernel family that made it."""
    arr, ix = gpu.upload(src), [gpu.upload(idx)]
    first = gpu.scatter_add(arr, ix, 1, [cells]).numpy()
    gpu.profile(1)
    again = gpu.scatter_add(arr, ix, 1, [cells]).numpy()
    labels = list(gpu.profile_report())
    gpu.profile(0)
    assert "scatter_counted" in labels, labels
    assert np.array_equal(first, again)
    return first


@pytest.mark.parametrize("dt", [np.float32, np.float64, np.int8])
@pytest.mark.parametrize("m,cells,hot,width", [(6000, 400, h, w) for h in (1, 3) for w in (1, 3, 40, 128, 301)] + [(140000, 3000, 2, w) for w in (1, 3, 40)])
def test_a_few_cells_take_half_of_the_hits(gpu, m, cells, hot, width, dt):
    """A padding index: runs of thousands beside ordinary ones (and a table of bits of either size)."""
    rng = np.random.default_rng(width + hot)
    idx = rng.integers(0, cells, m)
    idx[: m // 2] = rng.integers(0, hot, m // 2) * 7
    idx = rng.permutation(idx).astype(np.int64)
    shape = (m,) if width == 1 else (m, width)
    src = rng.integers(-100, 100, shape).astype(dt) if np.dtype(dt).kind == "i" else rng.standard_normal(shape).astype(dt)
    assert np.array_equal(counted(gpu, src, idx, cells), in_segments(src, idx, cells))


def test_all_positions_in_one_cell(gpu):
    rng = np.random.default_rng(14)
    m = 1 << 20
    src, idx = rng.standard_normal(m).astype(np.float32), np.full(m, 2047, np.int64)
    assert np.array_equal(counted(gpu, src, idx, 2048), in_segments(src, idx, 2048))


@pytest.mark.parametrize("dt", [np.float32, np.float64])
@pytest.mark.parametrize("cells,m,width", [(1, 1, 100003), (10, 32, 40000), (3, 300, 10001), (16, 16, 150528), (5, 64, 25004), (2, 65, 33), (4097, 2, 515), (7, 700, 2052), (3, 1500, 10001),
                                          (4, 1100, 30000), (1, 512, 7000), (9, 1025, 2051), (200, 1024, 129)])
def test_few_cells_with_wide_slices(gpu, cells, m, width, dt):
    rng = np.random.default_rng(cells + m)
    idx = rng.integers(-1, cells, m).astype(np.int64)
    src = rng.standard_normal((m, width)).astype(dt)
    inside = idx >= 0
    arr, ix = gpu.upload(src), [gpu.upload(idx)]
    assert np.array_equal(gpu.scatter_add(arr, ix, 1, [cells]).numpy(), in_segments(src[inside], idx[inside], cells))


@pytest.mark.parametrize("dt", [np.float32, np.float64])
@pytest.mark.parametrize("m,cells,width", [(100000, 400, 16), (131072, 300, 1), (131073, 300, 2), (131072, 4096, 3), (131072, 4095, 4), (9000, 20, 64), (70000, 140, 5), (1 << 20, 2100, 1),
                                           (1 << 20, 16000, 1), (16385, 256, 8), (4097, 64, 1)])
def test_many_cells_are_hit_often(gpu, m, cells, width, dt):
    """Dozens to hundreds of hits for every cell: either way of ordering long runs, and blocks that count 256 to 4096 positions."""
    rng = np.random.default_rng(m + cells)
    idx = rng.integers(0, cells, m).astype(np.int64)
    idx[rng.permutation(m)[: m // 50]] = 5            # (and one of thousands)
    src = rng.standard_normal((m,) if width == 1 else (m, width)).astype(dt)
    assert np.array_equal(counted(gpu, src, idx, cells), in_segments(src, idx, cells))


@pytest.mark.parametrize("dt", [np.float32, np.float64])
@pytest.mark.parametrize("cells,width", [(2000, 8), (60, 8), (60, 5)])
def test_positions_in_two_dims_that_do_not_merge(gpu, cells, width, dt):
    rng = np.random.default_rng(cells + width)
    idx, src = rng.integers(0, cells, (130, 77)).astype(np.int64), rng.standard_normal((77, 130, width)).astype(dt)
    out = gpu.scatter_add(gpu.upload(src).transpose([1, 0, 2]), [gpu.upload(idx)], 2, [cells]).numpy()
    assert np.array_equal(out, in_segments(np.ascontiguousarray(src.transpose(1, 0, 2)).reshape(-1, width), idx.reshape(-1), cells))

"""Zero-extensions wait (PadJob, csrc/ewise.hip): products that copy their operand to LDS read the array that is extended instead
(Extended, csrc/footprint.hip); everybody else finds the extension written."""
import numpy as np
import pytest

from conftest import capi, pkg
from test_contract_map import RELU

pytestmark = pytest.mark.gpu

O1, O2 = capi.OP1, capi.OP2


def source(ctx, x, how):
    """x [B, C, H, W] as an array that lies as it is, with the channels last, or amid a larger one."""
    if how == "plain":
        return ctx.upload(x)
    if how == "channels last":
        return ctx.upload(np.ascontiguousarray(x.transpose(0, 2, 3, 1))).transpose([0, 3, 1, 2])
    big = np.full((x.shape[0] + 2, x.shape[1], x.shape[2] + 1, x.shape[3] + 3), np.nan, x.dtype)
    big[1:-1, :, :-1, :-3] = x
    a = ctx.upload(big)
    for d, (first, n) in enumerate(zip((1, 0, 0, 0), x.shape)):
        a = a.slice(d, first, n)
    return a


def forward(ctx, p, ker, bias, H, Wd):
    """relu (conv + bias) of the extended p, its 2 x 2 maxima where they fit, as the first layers of a network ask for it."""
    (B, Ci), (Co, _, kh, kw), dt = p.shape[:2], ker.shape, ker.dtype
    sp = p.strides
    sh = [B, Co, H, Wd, Ci, kh, kw]
    a = p.as_strided(sh, [sp[0], 0, sp[2], sp[3], sp[1], sp[2], sp[3]], 0)
    b = ctx.upload(ker).as_strided(sh, [0, Ci * kh * kw, 0, 0, kh * kw, kw, 1], 0)
    kept = [B, Co, H, Wd]
    ins = [None, ctx.upload(bias).as_strided(kept, [0, 1, 0, 0], 0)] + [ctx.upload(np.asarray(v, dt)).as_strided(kept, [0, 0, 0, 0], 0) for v in (0, 1)]
    ext = None
    if H % 2 == 0 and Wd % 2 == 0:
        ext = (7, [B, Co, H // 2, Wd // 2, 2, 2], [Co * H * Wd, H * Wd, 2 * Wd, 2, Wd, 1], 2, True)
    outs, vals, idx = ctx.contract_map(a, b, 4, ins, RELU, [5, 7], ext)
    return outs + ([vals, idx] if ext else [])


def kernel_gradient(ctx, p, u, v, kh, kw):
    """sum over images and places of the extended p's windows times u * v, an expression."""
    (B, Ci), (Co, H, Wd) = p.shape[:2], u.shape[1:]
    sp = p.strides
    sh = [Co, Ci, kh, kw, B, H, Wd]
    a = p.as_strided(sh, [0, sp[1], sp[2], sp[3], sp[0], sp[2], sp[3]], 0)
    e = ctx.operand([ctx.upload(u), ctx.upload(v)], [(1, O2["mul"], 0, 0, 1, 0)], 2, [B, Co, H, Wd], (sh, [H * Wd, 0, 0, 0, Co * H * Wd, Wd, 1], 0))
    return [ctx.contract_operands(a, e, 4)]


@pytest.mark.parametrize("B,Ci,Co,H,W,k,dt,lo,how", [
    (300, 16, 16, 14, 14, 5, np.float64, 2, "plain"),
    (300, 16, 16, 14, 14, 5, np.float32, 2, "plain"),
    (260, 1, 16, 28, 28, 5, np.float64, 2, "plain"),
    (260, 1, 16, 28, 28, 5, np.float32, 2, "plain"),
    (130, 12, 12, 10, 14, 3, np.float64, 1, "plain"),      # one zero in front: element by element
    (130, 12, 12, 10, 14, 3, np.float32, 1, "plain"),
    (130, 12, 16, 9, 15, 5, np.float64, 2, "plain"),       # odd extents: no pooling, no vectors
    (130, 12, 16, 12, 12, 5, np.float64, 4, "plain"),      # all the zeros in front
    (130, 12, 16, 12, 12, 5, np.float64, 0, "plain"),      # ... or behind
    (130, 12, 16, 12, 16, 5, np.float32, 2, "channels last"),
    (130, 12, 16, 12, 16, 5, np.float64, 2, "channels last"),
    (130, 12, 16, 12, 16, 5, np.float64, 2, "slice"),
    (130, 12, 16, 12, 16, 5, np.float32, 2, "slice"),
    (9, 3, 4, 6, 8, 3, np.float64, 1, "plain"),            # too small to wait
])
def test_products_read_what_is_extended(gpu, B, Ci, Co, H, W, k, dt, lo, how):
    """The same bits as from an extension that somebody has read before."""
    rng = np.random.default_rng(B + k)
    x = rng.uniform(-1, 1, (B, Ci, H, W)).astype(dt)
    x[0, 0, 0, 0], x[-1, -1, -1, -1] = 0, -0.0
    ker, bias = rng.uniform(-0.4, 0.4, (Co, Ci, k, k)).astype(dt), rng.uniform(-0.4, 0.4, (Co,)).astype(dt)
    u, v = (rng.uniform(-1, 1, (B, Co, H, W)).astype(dt) for _ in range(2))
    lo, hi = [0, 0, lo, lo], [0, 0, k - 1 - lo, k - 1 - lo]
    s = source(gpu, x, how)

    def both(p):
        return forward(gpu, p, ker, bias, H, W) + kernel_gradient(gpu, p, u, v, k, k)

    written = s.pad(lo, hi)
    assert np.array_equal(written.numpy(), np.pad(x, list(zip(lo, hi))))
    want = [w.numpy() for w in both(written)]
    win = np.lib.stride_tricks.sliding_window_view(written.numpy().astype(np.float64), (k, k), axis=(2, 3))
    z = np.einsum("bihwpq,oipq->bohw", win, ker.astype(np.float64)) + bias.astype(np.float64)[None, :, None, None]
    mag = np.einsum("bihwpq,oipq->bohw", np.abs(win), np.abs(ker.astype(np.float64))) + 1
    assert np.all(np.abs(want[1] - np.maximum(z, 0)) <= np.finfo(dt).eps * (Ci * k * k + 4) * mag)
    gpu.profile(2)
    p = s.pad(lo, hi)
    got = both(p)
    del p
    got = [g.numpy() for g in got]
    labels = list(gpu.profile_report())
    gpu.profile(0)
    for g, w in zip(got, want):
        assert np.array_equal(g, w)
    if any("footprint" in n and ",map(" in n for n in labels) and any("footprint" in n and ",ymap" in n for n in labels):      # (else a product needs it written)
        assert not any(n.startswith("pad[") for n in labels), labels
    if Ci == 16:
        assert any("footprint" in n for n in labels) and not any(n.startswith("pad[") for n in labels), labels


@pytest.mark.parametrize("Ci,H,dt,written", [
    (16, 24, np.float32, False),      # 10,816 elements of an image, element by element: fits
    (16, 26, np.float32, True),       # 12,544: two loads a lane too many
    (32, 22, np.float32, True),       # ... by far
    (16, 22, np.float64, False),
])
def test_layers_whose_extension_does_not_fit(gpu, Ci, H, dt, written):
    """One zero in front, so the extension is staged element by element: where that is too much, the layer is still one kernel, over
    the written extension."""
    rng = np.random.default_rng(H)
    x = rng.uniform(-1, 1, (150, Ci, H, H)).astype(dt)
    ker, bias = rng.uniform(-0.4, 0.4, (16, Ci, 3, 3)).astype(dt), rng.uniform(-0.4, 0.4, (16,)).astype(dt)
    s = gpu.upload(x)
    p = s.pad([0, 0, 1, 1], [0, 0, 1, 1])
    gpu.sync()                            # written
    want = [o.numpy() for o in forward(gpu, p, ker, bias, H, H)]
    gpu.profile(2)
    got = [o.numpy() for o in forward(gpu, s.pad([0, 0, 1, 1], [0, 0, 1, 1]), ker, bias, H, H)]
    labels = list(gpu.profile_report())
    gpu.profile(0)
    for g, w in zip(got, want):
        assert np.array_equal(g, w)
    assert any("footprint" in n and ",map(" in n for n in labels) and not any(n == "argminmax" for n in labels), labels
    assert any(n.startswith("pad[") for n in labels) == written, labels


@pytest.mark.parametrize("dt", [np.float64, np.float32])
def test_others_find_the_extension_written(gpu, dt):
    rng = np.random.default_rng(2)
    x, y = (rng.uniform(-1, 1, (130, 12, 12, 16)).astype(dt) for _ in range(2))
    ker, bias = rng.uniform(-0.4, 0.4, (16, 12, 5, 5)).astype(dt), rng.uniform(-0.4, 0.4, (16,)).astype(dt)
    lo, hi = [0, 0, 2, 2], [0, 0, 2, 2]
    pad = lambda v: np.pad(v, list(zip(lo, hi)))
    s = gpu.upload(x)
    conv = lambda p: [o.numpy() for o in forward(gpu, p, ker, bias, 12, 16)]
    want = conv(gpu.upload(pad(x)))
    # an elementwise pass, a part of it, a product, and it itself
    p = s.pad(lo, hi)
    first = conv(p)
    assert np.array_equal(p.ewise1("neg").numpy(), -pad(x))
    assert np.array_equal(p.slice(2, 1, 3).numpy(), pad(x)[:, :, 1:4])
    assert np.array_equal(p.numpy(), pad(x))
    second = conv(p)
    for a, b, w in zip(first, second, want):
        assert np.array_equal(a, w) and np.array_equal(b, w)
    # what is extended changes: the extension is that of the values before
    p = s.pad(lo, hi)
    s.assign(gpu.upload(y))
    for a, w in zip(conv(p), want):
        assert np.array_equal(a, w)
    assert np.array_equal(p.numpy(), pad(x))
    # it goes away while its extension waits; an extension of an extension
    q = gpu.upload(x).pad(lo, hi)
    del s
    assert np.array_equal(q.pad(lo, hi).numpy(), pad(pad(x)))
    # more than may wait
    ps = [gpu.upload(x + dt(i)).pad(lo, hi) for i in range(7)]
    for i, p in enumerate(ps):
        assert np.array_equal(p.numpy(), pad(x + dt(i)))


def test_extensions_of_a_recording():
    """Values of a recording that are extensions are refreshed by every launch."""
    host = pkg.hostapi.Host()
    rng = np.random.default_rng(3)
    x, y = rng.uniform(-1, 1, (2, 200, 211))
    a = host.concrete(x)

    def program():
        wide = (a * 2.0 + 1.0).sgather((204, 215), lambda i, j: [i - 2, j - 2])
        return [wide, wide * wide, a.sgather((202, 213), lambda i, j: [i - 1, j - 1])]

    [v.numpy() for v in program()]
    graph, res = host.capture(program)
    try:
        for v in (x, y, x, x, y):
            a.overwrite(v)
            graph.launch()
            w = np.pad(v * 2.0 + 1.0, 2)
            for got, want in zip(res, (w, w * w, np.pad(v, 1))):
                assert np.array_equal(got.numpy(), want)
            [q.numpy() for q in program()]
    finally:
        graph.free()


@pytest.mark.parametrize("batch,h,w,k,c,dt,written", [
    (130, 28, 28, 5, 16, np.float64, 0),
    (130, 28, 28, 5, 16, np.float32, 0),
    (260, 20, 24, 3, 12, np.float64, None),
    (260, 16, 32, 5, 8, np.float32, None),
    (300, 32, 32, 5, 4, np.float64, None),
])
def test_gradients_of_convolutions(batch, h, w, k, c, dt, written):
    """The network's gradient against numpy's, recorded and not; `written`: extensions that the recording writes."""
    import ref_numpy
    import test_held_sums as held
    wl = pkg.workloads.c3_cnn(batch, pkg.capi.F64 if dt == np.float64 else pkg.capi.F32, h, w, k, c, 32)
    host = pkg.hostapi.Host()
    ps, ds = wl.upload(host)
    program = lambda: (lambda loss, grads: [loss] + grads)(*wl.gradient(host, ps, ds))
    eager = [v.numpy() for v in program()]
    loss, grads = ref_numpy.cnn([p.astype(np.float64) for p in wl.params], *[d.astype(np.float64) for d in wl.data])
    tol = 1e-11 if dt == np.float64 else 1e-4      # (single precision: an arg-maximum or a relu near its edge goes the other way)
    for got, want in zip(eager, [np.asarray(loss)] + list(grads)):
        assert np.max(np.abs(got - want)) <= tol * np.max(np.abs(want))
    graph, res, labels = held.recorded(host, program)
    pads = [n for n in labels if n.startswith("pad[")]
    if written is not None:
        assert len(pads) == written and any(n.startswith("onehot") for n in labels), labels
    try:
        for _ in range(3):
            graph.launch()
            host.sync()
            for got, want in zip(res, eager):
                assert np.max(np.abs(got.numpy() - want)) <= (1e-12 if dt == np.float64 else 1e-5) * np.max(np.abs(want))
            [v.numpy() for v in program()]
    finally:
        graph.free()

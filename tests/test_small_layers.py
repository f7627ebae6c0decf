"""Layers of fewer than a million multiplications: the products and the program over their sum are one launch whatever the
size (csrc/smallk.hip), and the steps of a small recurrence one chain (csrc/smallk_chain.hpp)."""
import numpy as np
import pytest

from test_contract_sum_map import O1, O2, layer_case, matmul_views
import test_smallk_chain as chain

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dt", [np.float64, np.float32])
@pytest.mark.parametrize("m,n,ks,layouts", [
    (4, 16, [2, 2], ["mk", "mk"]),        # the smallest
    (16, 16, [4], ["mk"]),                # the smallest of a single product
    (5, 17, [2, 3], ["mk", "km"]),        # ragged everywhere, no vectors
    (64, 32, [10], ["km"]),               # the cotangent under a readout
    (33, 31, [29, 33], ["mk", "mk"]),
    (300, 16, [3, 2], ["km", "mk"]),
    (16, 999, [61], ["mk"]),              # just below a million
])
def test_layers(gpu, dt, m, n, ks, layouts):
    gpu.check(gpu.lib.profile_enable(gpu.h, 2))
    terms, ins, prog, slots, want = layer_case(gpu, dt, m, n, ks, layouts)
    got = gpu.contract_sum_map(terms, 2, ins, prog, slots)[0].numpy()
    labels = gpu.profile_report()
    gpu.check(gpu.lib.profile_enable(gpu.h, 0))
    assert sum(v[0] for k, v in labels.items()) == 1 and all("wholeK" in k for k in labels), labels
    assert got.dtype == dt and np.max(np.abs(got - want)) <= chain.step_bound(dt, ks)


@pytest.mark.parametrize("dt", [np.float64, np.float32])
@pytest.mark.parametrize("width,batch,k_in,steps,layers", [(32, 32, 28, 9, 2), (16, 16, 3, 8, 2), (50, 37, 28, 12, 2), (80, 64, 9, 8, 1)])
def test_small_recurrences_are_chains(gpu, dt, width, batch, k_in, steps, layers):
    chain.test_recurrence_forward(gpu, dt, width, batch, k_in, steps, layers)
    chain.test_recurrence_backward(gpu, dt, width, batch, steps)


def rounded_once(got, want, mag, k, also=0.0):
    """Sums of k exact products in fp64, in any order, rounded once to fp32 (and `also` behind that)."""
    return np.all(np.abs(got - want) <= 2.0 ** -24 * np.abs(want) + 2 * k * 2.0 ** -53 * mag + also + 2.0 ** -150)


SMALL = [
    (16, 16, [4], ["mk"]),
    (10, 250, [128], ["mk"]),             # a readout
    (128, 150, [10], ["km"]),             # the cotangent under it
    (33, 31, [29, 33], ["mk", "km"]),
    (40, 600, [28], ["mk"]),
    (130, 500, [13], ["km"]),             # more tiles of 16 x 16 than CUs: larger ones
    (16, 16, [1000], ["mk"]),             # K shared out between blocks: partial sums are fp64, too
    (9, 40, [700, 300], ["km", "mk"]),
]


# (a product alone, no program behind it, is another kernel's below a million multiplications)
@pytest.mark.parametrize("m,n,ks,layouts,form", [s + (f,) for s in SMALL for f in ("program", "bias", "sum") if f != "sum" or len(s[2]) > 1])
def test_small_fp32_sums_are_fp64(gpu, m, n, ks, layouts, form):
    rng = np.random.default_rng(m * n + len(ks))
    terms, want, mag = [], np.zeros((m, n)), np.zeros((m, n))
    for k, lay in zip(ks, layouts):
        w, x = rng.uniform(-1, 1, (m, k)).astype(np.float32), rng.uniform(-1, 1, (k, n)).astype(np.float32)
        wa = gpu.upload(w) if lay == "mk" else gpu.upload(np.ascontiguousarray(w.T)).transpose([1, 0])
        terms.append(matmul_views(wa, gpu.upload(x)))
        want += w.astype(np.float64) @ x.astype(np.float64)
        mag += np.abs(w).astype(np.float64) @ np.abs(x).astype(np.float64)
    b = rng.uniform(-1, 1, m).astype(np.float32)
    ins, prog, slots = {"program": ([None], [(0, O1["neg"], 0, 0, 0, 0)], [1]),
                        "bias": ([gpu.upload(b).replicate([n]).transpose([1, 0]), None], [(1, O2["sub"], 0, 1, 0, 0)], [2]),
                        "sum": ([None], [], [0])}[form]
    gpu.profile(2)
    got = gpu.contract_sum_map(terms, 2, ins, prog, slots)[0].numpy().astype(np.float64)
    labels = gpu.profile_report()
    gpu.profile(0)
    assert all("wholeK" in k and "sums64" in k for k in labels), labels
    if form == "bias":
        d = want - b[:, None].astype(np.float64)
        assert rounded_once(got, d, mag, sum(ks), 2.0 ** -24 * np.abs(want) * (1 + 2.0 ** -20))
    else:
        assert rounded_once(-got if form == "program" else got, want, mag, sum(ks))


@pytest.mark.parametrize("width,batch,k_in,steps", [(32, 64, 28, 9), (16, 16, 3, 8), (50, 37, 28, 12), (80, 61, 9, 8)])
def test_small_fp32_recurrences_add_in_fp64(gpu, width, batch, k_in, steps):
    """s_t = -(W x_t + V s_(t-1)) and its second layer: every step compared with fp64 on the results the device gave before it."""
    rng = np.random.default_rng(width)
    f = np.float32
    w = [rng.uniform(-1, 1, (width, k)).astype(f) for k in (k_in, width)]
    v = [(rng.uniform(-1, 1, (width, width)) * 2 / width ** 0.5).astype(f) for _ in range(2)]
    xs = [rng.uniform(-1, 1, (k_in, batch)).astype(f) for _ in range(steps)]
    neg = [(0, O1["neg"], 0, 0, 0, 0)]

    def work():
        up = gpu.upload
        zero, xa, params = up(np.zeros((), f)).replicate([batch]).replicate([width]), [up(x) for x in xs], [(up(a), up(b)) for a, b in zip(w, v)]
        layers = []
        for wa, va in params:
            s = []
            for t in range(steps):
                x = xa[t] if not layers else layers[0][t]
                s.append(gpu.contract_sum_map([matmul_views(wa, x), matmul_views(va, s[-1] if s else zero)], 2, [None], neg, [1])[0])
            layers.append(s)
        return [[a.numpy().astype(np.float64) for a in s] for s in layers]

    out, n, labels = chain.chains(gpu, work)
    assert n == 1, labels
    for layer in range(2):
        for t in range(steps):
            x = xs[t].astype(np.float64) if layer == 0 else out[0][t]
            s = out[layer][t - 1] if t else np.zeros((width, batch))
            a, b = w[layer].astype(np.float64), v[layer].astype(np.float64)
            want, mag = a @ x + b @ s, np.abs(a) @ np.abs(x) + np.abs(b) @ np.abs(s)
            assert rounded_once(-out[layer][t], want, mag, 2 * width + k_in), (layer, t)


@pytest.mark.parametrize("width,batch,steps", [(128, 150, 9), (100, 130, 10)])
def test_a_small_product_in_a_chain_of_large_ones(gpu, width, batch, steps):
    """d_t = (V^T d_(t+1)) * g_t under a readout of ten classes: the first product alone has fewer than a million multiplications,
    and alone adds in fp64."""
    rng = np.random.default_rng(width)
    f = np.float32
    v, wo, dl = (rng.uniform(-1, 1, s).astype(f) for s in ((width, width), (10, width), (10, batch)))
    g = rng.uniform(0.1, 0.2, (width, batch)).astype(f)
    mul = [(1, O2["mul"], 0, 0, 1, 0)]

    def work():
        va, wa, d, ga, res = gpu.upload(v).transpose([1, 0]), gpu.upload(wo).transpose([1, 0]), gpu.upload(dl), gpu.upload(g), []
        for t in range(steps):
            d = gpu.contract_sum_map([matmul_views(va if t else wa, d)], 2, [None, ga], mul if t else [(0, O1["neg"], 0, 0, 0, 0)], [2])[0]
            res.append(d)
        return [a.numpy().astype(np.float64) for a in res]

    out, n, labels = chain.chains(gpu, work)
    assert n == 1, labels
    w64, v64, g64 = wo.astype(np.float64), v.astype(np.float64), g.astype(np.float64)
    assert rounded_once(-out[0], w64.T @ dl, np.abs(w64).T @ np.abs(dl).astype(np.float64), 10)
    for t in range(1, steps):
        mag = np.abs(v64).T @ np.abs(out[t - 1]) * g64
        assert np.all(np.abs(out[t] - (v64.T @ out[t - 1]) * g64) <= (width + 3) * 2.0 ** -24 * mag), t

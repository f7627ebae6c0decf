"""What users of the backend have it do, as timed cases: gradients of whole objectives.

A case is one gradient program (value and reverse pass) of a family at a size, in an
element type and in one of the three ways a program submits it:

  recorded   the program is recorded once and every pass is one launch of it: evaluating
             a gradient artifact again and again (what training and benchmarking do)
  eager      every pass submits the program operation by operation and reads the
             objective's value back (a new objective at every step, interactive use)
  train      recorded, with the Adam update and the write-back of parameters and moments

The families are the objectives the package brings (`horde-ad_amd/workloads.py`) and the
lookup of table rows by an index vector, whose reverse pass is the general scatter-add:

  elementwise   sum (atan2 z (x * sin y) + z * (x * sin y)) w.r.t. three matrices
  dense         dense network with tanh or relu, softmax cross entropy, w.r.t. all weights
  conv          two layers of convolution + relu + 2x2 pooling, two dense layers
  recurrent     two-layer tanh recurrence over a sequence, readout of the last state
  lookup        sum (rows of a table picked by data * weights) w.r.t. the table
"""
import math

import numpy as np

import __graft_entry__ as entry

pkg = entry.load_package()
capi, H, W, OPT = pkg.capi, pkg.hostapi, pkg.workloads, pkg.optimizer

DTYPE = {"f64": capi.F64, "f32": capi.F32}
SIZE = {"f64": 8, "f32": 4}
_host = None


def host():
    """The one context a process keeps."""
    global _host
    if _host is None:
        _host = H.Host()
    return _host


def listed():
    return [
        # the smallest calls: a few thousand elements, all of it host work and launches
        dict(name="elementwise_tiny_eager", kind="elementwise", n=64, m=48, dtype="f64", mode="eager"),
        # an odd, mid-sized elementwise objective
        dict(name="elementwise_odd_f32", kind="elementwise", n=1003, m=1021, dtype="f32", mode="recorded"),
        # the benchmark's elementwise objective: 400 MB in, 400 MB out
        dict(name="elementwise_large", kind="elementwise", n=4096, m=4096, dtype="f64", mode="recorded"),
        # a ragged minibatch through the MNIST dense network, submitted as it is written
        dict(name="dense_minibatch_eager", kind="dense", batch=130, widths="784,300,100,10", act="tanh", dtype="f64", mode="eager"),
        # the MNIST dense network on a large batch (the benchmark's)
        dict(name="dense_fcnn", kind="dense", batch=5000, widths="784,300,100,10", act="tanh", dtype="f64", mode="recorded"),
        # wide dense network (the benchmark's): matrix products all through
        dict(name="dense_wide", kind="dense", batch=8192, widths="784,2048,2048,10", act="relu", dtype="f32", mode="recorded"),
        # the small CNN of the reference's own benchmark: 24x24, four channels, batch of 7
        dict(name="conv_tiny_eager", kind="conv", batch=7, h=24, w=24, ksize=3, c_out=4, n_hidden=5, dtype="f64", mode="eager"),
        # the MNIST CNN, one gradient of a batch of 1000 (the benchmark's headline)
        dict(name="conv_mnist", kind="conv", batch=1000, h=28, w=28, ksize=5, c_out=16, n_hidden=128, dtype="f64", mode="recorded"),
        # the same network trained in single precision on an odd minibatch
        dict(name="conv_train_f32", kind="conv", batch=250, h=28, w=28, ksize=5, c_out=16, n_hidden=128, dtype="f32", mode="train"),
        # the MNIST RNN, sequences of 28 rows (the benchmark's)
        dict(name="recurrent_mnist", kind="recurrent", batch=5000, steps=28, n_in=28, width=128, dtype="f32", mode="recorded"),
        # the same network on a minibatch in double precision
        dict(name="recurrent_minibatch_f64", kind="recurrent", batch=150, steps=28, n_in=28, width=128, dtype="f64", mode="recorded"),
        # rows of a table picked by data and their adjoint, the sorted scatter-add
        dict(name="lookup_rows", kind="lookup", rows=20000, width=128, picks=100000, dtype="f32", mode="eager"),
    ]


def _log(rng, lo, hi):
    """A whole number between lo and hi, spread over its logarithm."""
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    while True:
        kind = rng.choice(["elementwise", "dense", "conv", "recurrent", "lookup"])
        dtype = rng.choice(["f64", "f32"])
        mode = rng.choice(["recorded", "recorded", "eager"])
        if kind == "elementwise":
            c = dict(kind=kind, n=_log(rng, 30, 4096), m=_log(rng, 30, 4096), dtype=dtype, mode=mode)
        elif kind == "dense":
            hidden = [_log(rng, 64, 2048) for _ in range(2)]
            c = dict(kind=kind, batch=_log(rng, 32, 8192), widths=",".join(str(v) for v in [784] + hidden + [10]),
                     act=rng.choice(["tanh", "relu"]), dtype=dtype, mode=rng.choice(["recorded", "eager", "train"]))
        elif kind == "conv":
            c = dict(kind=kind, batch=_log(rng, 5, 1000), h=rng.choice([16, 20, 24, 28, 32]), w=rng.choice([16, 20, 24, 28, 32]), ksize=rng.choice([3, 5]),
                     c_out=rng.choice([4, 8, 12, 16]), n_hidden=_log(rng, 16, 256), dtype=dtype, mode=rng.choice(["recorded", "eager", "train"]))
        elif kind == "recurrent":
            c = dict(kind=kind, batch=_log(rng, 32, 5000), steps=rng.randint(8, 28), n_in=28, width=_log(rng, 32, 160), dtype=dtype, mode=mode)
        else:
            c = dict(kind=kind, rows=_log(rng, 500, 200000), width=_log(rng, 1, 256), picks=_log(rng, 1000, 200000), dtype=dtype, mode=mode)
        # nothing dearer than the largest listed case: a double-precision operation takes about twice as long
        if work(c)["flops"] * (2 if dtype == "f64" else 1) <= 2.5e11:
            return c


def _widths(case):
    return [int(v) for v in case["widths"].split(",")]


def _initial(seed, params, dtype):
    """Initial weights and biases of a layered network: uniform, scaled by the layer's fan-in
    (the objective's exponentials are taken unshifted from above: single precision needs logits of order one)."""
    bound = [math.sqrt(3.0 / (p.size // p.shape[0])) for p in params[0::2]]
    return [W.uniform(seed + k, p.shape, -bound[k // 2], bound[k // 2], dtype) for k, p in enumerate(params)]


def _workload(case, seed):
    """The objective with its inputs drawn from the seed."""
    dtype, kind = DTYPE[case["dtype"]], case["kind"]
    base = 1000 * seed
    if kind == "elementwise":
        def away(a):
            return np.where(np.abs(a) < 0.1, np.where(a < 0, a - 0.1, a + 0.1), a).astype(W.NP[dtype])
        wl = W.c0_elementwise(1, 1, dtype)
        x, y, z = (W.uniform(base + k, (case["n"], case["m"]), -2, 2, dtype) for k in range(3))
        wl.params = [away(x), y, away(z)]
    elif kind == "dense":
        widths = _widths(case)
        make = W.c1_fcnn if case["act"] == "tanh" else W.c2_wide
        wl = make(case["batch"], dtype, widths)
        wl.data = [W.pixels(base, (widths[0], case["batch"]), dtype), W.one_hot_labels(base + 1, widths[-1], case["batch"], dtype)]
        wl.params = _initial(base + 2, wl.params, dtype)
    elif kind == "conv":
        wl = W.c3_cnn(case["batch"], dtype, case["h"], case["w"], case["ksize"], case["c_out"], case["n_hidden"])
        wl.data = [W.pixels(base, wl.data[0].shape, dtype), W.one_hot_labels(base + 1, 10, case["batch"], dtype)]
        wl.params = _initial(base + 2, wl.params, dtype)
    elif kind == "recurrent":
        wl = W.c4_rnn(case["batch"], dtype, case["steps"], case["n_in"], case["width"])
        wl.data = [W.pixels(base, wl.data[0].shape, dtype), W.one_hot_labels(base + 1, 10, case["batch"], dtype)]
        wl.params = [W.uniform(base + 2 + k, p.shape, -0.1, 0.1, dtype) for k, p in enumerate(wl.params)]
    else:
        rows, width, picks = case["rows"], case["width"], case["picks"]
        ix = np.random.Generator(np.random.Philox(base)).integers(0, rows, picks)

        def objective(ps, ds):
            index, weights = ds
            picked = ps[0].sgather((picks,), lambda i: [index.sindex0([i])])
            return (picked * weights).ssum0()

        wl = W.Workload("lookup", dtype, picks, [W.uniform(base + 1, (rows, width), -1, 1, dtype)],
                        [ix, W.uniform(base + 2, (picks, width), -1, 1, dtype)], objective, 0.0, None)
    return wl


class Arrays(dict):
    """Arrays that stay on the device: looking one up copies it to the host."""

    def __getitem__(self, key):
        return super().__getitem__(key).numpy()


class State:
    """The uploaded inputs of a case and, where it is recorded, the recording."""

    def __init__(self, case, seed):
        self.mode, self.graph, h, wl = case["mode"], None, host(), _workload(case, seed)
        ps, ds = wl.upload(h)
        np_type = W.NP[wl.dtype]
        wl.params = wl.data = None

        def gradient():
            return wl.gradient(h, ps, ds)

        self.program = gradient
        if self.mode == "train":
            ms, vs = [[h.concrete(np.zeros(p.shape, np_type)) for p in ps] for _ in range(2)]
            self.np_type, self.step = np_type, 1
            self.alphat = alphat = h.concrete(step_size(1, np_type))

            def train():
                loss, grads = gradient()
                new = OPT.adamApply(OPT.defaultArgsAdam, alphat, ms, vs, ps, grads)
                for dst, src in zip(ms + vs + ps, new[0] + new[1] + new[2]):
                    dst.assign(src)
                return loss, grads

            self.program = train
        if self.mode != "eager":
            self.program()                       # the program's constants are made by an eager run
            self.graph, (loss, grads) = h.capture(self.program)
            self.out = Arrays(loss=loss, **{"gradient%d" % i: g for i, g in enumerate(grads)})
            if self.mode == "train":
                self.out.update({"parameter%d" % i: p for i, p in enumerate(ps)})

    def __del__(self):
        if self.graph is not None:
            self.graph.free()


def step_size(t, np_type):
    """Adam's step size at iteration t."""
    a = OPT.defaultArgsAdam
    return np.array(a.alpha * math.sqrt(1 - a.betaTwo ** t) / (1 - a.betaOne ** t), np_type)


def prepare(case, seed):
    return State(case, seed)


def run(state):
    if state.mode == "eager":
        loss, grads = state.program()
        value = float(loss.numpy())
        return [value, Arrays({"gradient%d" % i: g for i, g in enumerate(grads)})]
    if state.mode == "train":
        state.step += 1
        state.alphat.overwrite(step_size(state.step, state.np_type))
    state.graph.launch()
    return state.out


def work(case):
    """Operations of the mathematics (matrix products for the networks, about 20 per element for
    the elementwise objective) and the inputs read and gradients written once."""
    size, kind = SIZE[case["dtype"]], case["kind"]
    if kind == "elementwise":
        elements = case["n"] * case["m"]
        return {"bytes": 6.0 * size * elements, "flops": 20.0 * elements}
    if kind == "lookup":
        moved = case["picks"] * case["width"]
        # the rows that are picked, the weights, the index vector, and the whole gradient
        return {"bytes": float(size * (2 * moved + case["rows"] * case["width"]) + 8 * case["picks"]), "flops": 3.0 * moved}
    b = float(case["batch"])
    if kind == "dense":
        widths = _widths(case)
        mm = sum(i * o for i, o in zip(widths[:-1], widths[1:]))
        flops = 2.0 * b * (2 * mm + sum(i * o for i, o in zip(widths[1:-1], widths[2:])))
        n_par, n_in = mm + sum(widths[1:]), b * (widths[0] + widths[-1])
    elif kind == "conv":
        h, w, c, k2 = case["h"], case["w"], case["c_out"], case["ksize"] ** 2
        flat, hidden = c * (h // 4) * (w // 4), case["n_hidden"]
        conv1, conv2 = 2 * b * c * h * w * k2, 2 * b * c * c * (h // 2) * (w // 2) * k2
        flops = 2 * conv1 + 3 * conv2 + 3 * 2 * b * hidden * (flat + 10)
        n_par, n_in = c * k2 + c + c * c * k2 + c + hidden * flat + hidden + 10 * hidden + 10, b * (h * w + 10)
    else:
        width, n_in_step, steps = case["width"], case["n_in"], case["steps"]
        flops = 3 * steps * 2 * b * (width * n_in_step + 3 * width * width) + 3 * 2 * b * 10 * width
        n_par, n_in = width * n_in_step + 3 * width * width + 2 * width + 10 * width + 10, b * (steps * n_in_step + 10)
    # parameters in, gradients out; training also reads and writes two moments and the parameters
    passes = 7 if case["mode"] == "train" else 2
    return {"bytes": float(size * (passes * n_par + n_in)), "flops": float(flops)}


def tolerance(case):
    """Double precision against the same programs with every operation run by itself (other orders of
    summation): at most 2e-15 of the result; an objective that nearly cancels loses two or three digits more.
    Single precision against double on the same inputs: at most 4e-7, but where relu or an arg-maximum
    decides, a unit near the edge may go the other way (wide dense network: 4e-5, single elements 2e-3)."""
    if case["dtype"] == "f64":
        return {"rel": 1e-12}
    if case["kind"] == "conv" or case.get("act") == "relu":
        return {"rel": 2e-4, "max": 1e-2}
    # an objective that is one sum over all elements loses what it cancels
    return {"rel": 1e-5 if case["kind"] in ("elementwise", "lookup") else 2e-6}

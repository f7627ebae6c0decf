"""Sums of short products with few 16 x 16 tiles: a block loads its operands whole and its wavefronts share K out
(csrc/smallk.hip, choose_flat)."""
import numpy as np
import pytest

from conftest import capi
from test_contract_sum_map import layer_case

pytestmark = pytest.mark.gpu

O1, O2 = capi.OP1, capi.OP2


@pytest.mark.parametrize("dt", [np.float64, np.float32])
@pytest.mark.parametrize("m,n,ks,layouts,flat", [
    (128, 150, [28, 128], ["mk", "mk"], True),
    (128, 150, [128, 128], ["km", "km"], True),
    (128, 512, [128, 128], ["mk", "km"], True),              # 256 tiles: the last size for 256 CUs
    (128, 513, [128, 128], ["mk", "km"], False),
    (17, 1000, [70], ["mk"], True),                          # two rows of tiles, the second one row high
    (33, 131, [250], ["km"], True),                          # ragged everywhere, odd extents: no vectors
    (4, 2000, [129], ["mk"], True),                          # the fewest rows; k one over a whole number of quarters
    (128, 75, [2, 3, 127, 15], ["mk", "km", "mk", "km"], True),
    (100, 130, [300], ["mk"], True),
    (64, 130, [700], ["mk"], False),                         # operands too large to stand in LDS whole
])
def test_layers(gpu, dt, m, n, ks, layouts, flat):
    if dt == np.float32 and ks == [700]:
        ks = [1000]
    eps = np.finfo(dt).eps
    for bias in (True, False):
        gpu.check(gpu.lib.profile_enable(gpu.h, 2))
        terms, ins, prog, slots, want = layer_case(gpu, dt, m, n, ks, layouts, bias)
        got = gpu.contract_sum_map(terms, 2, ins, prog, slots)[0].numpy()
        labels = list(gpu.profile_report())
        gpu.check(gpu.lib.profile_enable(gpu.h, 0))
        assert any(",t16x16," in k for k in labels) == flat, labels
        # |w| <= 0.3, |x| <= 1: a rounding per product and per addition, and tanh (slope at most 1) with two units of its own
        bound = eps * (0.3 * sum(ks) * (sum(ks) + 8) + 4)
        assert got.dtype == dt and np.max(np.abs(got - want)) <= bound


@pytest.mark.parametrize("dt", [np.float64, np.float32])
def test_program_over_full_row_and_column_inputs(gpu, oracle, dt):
    """Inputs that run along both dims, along one, along none and transposed; two results, one of them a comparison."""
    rng = np.random.default_rng(3)
    m, n, k = 100, 141, 90
    x = {"w": rng.uniform(-0.3, 0.3, (m, k)), "x": rng.uniform(-1, 1, (k, n)), "h": rng.uniform(-1, 1, (m, n)), "t": rng.uniform(-1, 1, (n, m)),
         "row": rng.uniform(-1, 1, (n,)), "col": rng.uniform(-1, 1, (m,)), "one": np.asarray(0.25)}
    res = []
    for ctx in (gpu, oracle):
        u = {key: ctx.upload(v.astype(dt)) for key, v in x.items()}
        a, b = u["w"].replicate([n]).transpose([1, 0]), u["x"].replicate([m]).transpose([0, 2, 1])
        ins = [u["h"], None, u["t"].transpose([1, 0]), u["row"].replicate([m]), u["col"].replicate([n]).transpose([1, 0]), u["one"].replicate([m, n])]
        prog = [(1, O2["mul"], 0, 0, 1, 0), (1, O2["add"], 0, 6, 2, 0), (1, O2["mul"], 0, 7, 3, 0), (1, O2["sub"], 0, 8, 4, 0), (1, O2["mul"], 0, 9, 5, 0),
                (2, capi.CMP["lt"], 0, 9, 0, 0)]
        res.append([o.numpy() for o in ctx.contract_sum_map([(a, b)], 2, ins, prog, [10, 11, 1])])
    scale = np.max(np.abs(res[1][0]))
    tol = 1e-12 if dt == np.float64 else 1e-5
    assert np.max(np.abs(res[0][0] - res[1][0])) <= tol * scale
    assert np.max(np.abs(res[0][2] - res[1][2])) <= tol * np.max(np.abs(res[1][2]))
    assert np.mean(res[0][1] != res[1][1]) <= 1e-3       # (ties of the comparison)


@pytest.mark.parametrize("dt", [np.float64, np.float32])
@pytest.mark.parametrize("m,n,ks,layouts", [(100, 130, [301], ["mk"]), (40, 75, [623], ["mk"]), (131, 75, [302], ["km"]), (60, 200, [303], ["mk"]), (100, 200, [33, 101], ["mk", "mk"]), (100, 200, [31, 99], ["mk", "mk"]),
                                            (17, 1000, [131, 66], ["mk", "km"]), (64, 130, [67, 5, 130], ["mk", "mk", "km"])])
def test_k_of_no_whole_number_of_vectors(gpu, dt, m, n, ks, layouts):
    """Operands with k side by side: whole vectors in one chunk, one to three elements in another; and products of two such."""
    test_layers(gpu, dt, m, n, ks, layouts, dt == np.float32 or ks[0] < 312)
    rng = np.random.default_rng(m)
    x, y = rng.uniform(-1, 1, (m, ks[0])).astype(dt), rng.uniform(-1, 1, (n, ks[0])).astype(dt)
    got = gpu.upload(x).replicate([n]).transpose([1, 0, 2]).contract(gpu.upload(y).replicate([m]), 2).numpy()
    # (a rounding per product and per addition)
    assert np.max(np.abs(got - x.astype(np.float64) @ y.astype(np.float64).T)) <= np.finfo(dt).eps * ks[0] * (ks[0] + 8) / 2

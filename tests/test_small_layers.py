"""Layers of fewer than a million multiplications: the products and the program over their sum are one launch whatever the
size (csrc/smallk.hip), and the steps of a small recurrence one chain (csrc/smallk_chain.hpp)."""
import numpy as np
import pytest

from test_contract_sum_map import layer_case
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

"""hgpu_contract_sum of many small products: together they are worth the matrix cores (csrc/gemm.hip, try_gemm)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dt", [np.float64, np.float32])
@pytest.mark.parametrize("m,n,k,terms", [(128, 28, 150, 28), (128, 28, 151, 27), (40, 33, 60, 32), (17, 16, 31, 33), (100, 90, 20, 12), (300, 7, 33, 30)])
@pytest.mark.parametrize("lay", ["KK", "RR"])
def test_terms_that_are_slices(gpu, dt, m, n, k, terms, lay):
    """The terms are slices of one array each, so an odd slice starts off a 16-byte boundary."""
    rng = np.random.default_rng(m + n + k)
    x, y = rng.uniform(-1, 1, (terms, m, k)).astype(dt), rng.uniform(-1, 1, (terms, n, k)).astype(dt)
    if lay == "KK":
        a, b = gpu.upload(x), gpu.upload(y)
    else:
        a, b = (gpu.upload(np.ascontiguousarray(v.transpose(0, 2, 1))).transpose([0, 2, 1]) for v in (x, y))
    pairs = [(a.index_prefix([t]).replicate([n]).transpose([1, 0, 2]), b.index_prefix([t]).replicate([m])) for t in range(terms)]
    got = gpu.contract_sum(pairs, 2).numpy()
    xd, yd = x.astype(np.float64), y.astype(np.float64)
    want = np.einsum("tmk,tnk->mn", xd, yd)
    # one rounding per product and one per addition, of the sum of magnitudes
    bound = np.finfo(dt).eps * (terms * k + 8) * np.einsum("tmk,tnk->mn", np.abs(xd), np.abs(yd))
    assert got.dtype == dt and np.all(np.abs(got - want) <= bound)

"""Reductions with few results and long chains: column sums, and the weight gradient of a first layer with a few filters,
whose pixels are cut into hundreds of partial results."""
import numpy as np
import pytest

import oracle
from util import he_normal, rel_l2

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("m,n", [(1, 1), (15, 17), (16, 16), (17, 1000), (127, 10), (129, 33), (1024, 5)])
def test_column_sums(gpu, m, n):
    a = np.random.default_rng(m + n).standard_normal((m, n)).astype(np.float32)
    got = gpu.kernels.colsum(gpu.to_device(a)).numpy().reshape(-1)
    # float64 sums rounded once: half an ulp of the result, and nothing for the order
    np.testing.assert_allclose(got, a.astype(np.float64).sum(0), rtol=2.0 ** -23, atol=1e-12)


@pytest.mark.parametrize("n,k,size", [(3, 4, 28), (64, 8, 28), (256, 8, 28), (40, 17, 33)])
@pytest.mark.parametrize("accumulate", [False, True])
def test_weight_gradient_of_few_filters(gpu, n, k, size, accumulate):
    rng = np.random.default_rng(n + k)
    x = rng.standard_normal((n, 1, size, size)).astype(np.float32)
    w, b = he_normal(rng, (k, 1, 2, 2)), rng.standard_normal((k,)).astype(np.float32)
    dy = rng.standard_normal((n, k, size - 1, size - 1)).astype(np.float32)
    dw0, db0 = (w, b) if accumulate else (np.zeros_like(w), np.zeros_like(b))
    _, col = oracle.conv2d_fwd(x, w, b, (1, 1), 0)
    _, dw_ref, db_ref = oracle.conv2d_bwd(dy, x.shape, w, col, (1, 1), 0, np.zeros_like(x), dw0.copy(), db0.copy())
    gw, gb = gpu.to_device(dw0), gpu.to_device(db0)
    gpu.kernels.conv2d_bwd_weight(gpu.to_device(dy), gpu.to_device(x), w.shape, (1, 1), 0, dw=gw, db=gb, accumulate=accumulate)
    assert rel_l2(gw.numpy(), dw_ref) <= 1e-5 and rel_l2(gb.numpy(), db_ref) <= 1e-5       # the fp32 path's bar

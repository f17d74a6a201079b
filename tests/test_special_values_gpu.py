"""Infinities in the adjoint's operands: with positive operands no sum has a NaN, and an infinite value makes exactly the
gradients infinite that it enters, also where it lies in the fiber that lanes past the last one repeat."""
import numpy as np
import pytest

import oracle
from kronmult993_amd import workloads as W
from kronmult993_amd.device import DeviceBatch

pytestmark = pytest.mark.gpu

SHAPES = [(2, 3), (3, 5), (3, 6), (3, 7), (4, 3), (4, 4), (4, 5), (4, 6), (4, 7), (4, 8), (5, 3), (5, 4), (5, 5), (6, 2),
          (6, 3), (6, 4)]
# a gradient sums at most n^d products of chains of d - 1 sums of n terms, all positive: (n^d + d n) roundings of u,
# each relative to the sum; the largest here is 4096 + 24
RTOL = {np.dtype(np.float64): 5000 * 2.0 ** -53, np.dtype(np.float32): 5000 * 2.0 ** -24}


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("d,n", SHAPES)
@pytest.mark.parametrize("where", ["x", "g"])
def test_adjoint_infinities(gpu, d, n, dtype, where):
    rng = np.random.default_rng(600 + 9 * d + n)
    nb, size, k = 5, n ** d, np.arange(5)
    x, g = rng.uniform(0.5, 1, nb * size), rng.uniform(0.5, 1, nb * size)
    (x if where == "x" else g)[3 * size - 1] = np.inf  # the last element of entry 2: the last fiber of every mode
    mats = rng.uniform(0.1, 1, nb * d * n * n) / n
    b = W.HostBatch(f"inf_{where}_d{d}n{n}", d, n, n, mats, np.arange(nb * d) * n * n, x, k * size, nb, k,
                    grad_out_pool=g).astype(dtype)
    print(f"[adjoint] {b.name} {b.dtype}", flush=True)
    db = DeviceBatch(b, device=str(gpu))
    db.adjoint_setup()
    db.run_adjoint()
    for got, ref in zip(db.gradients(), oracle.adjoint(b.astype(np.float64))):
        assert not np.isnan(ref).any()
        np.testing.assert_allclose(got.astype(np.float64), ref, rtol=RTOL[b.dtype])

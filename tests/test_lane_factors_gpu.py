"""FP32 sweeps of n = 4 and 8 on the matrix cores, factors held in the lanes: bit for bit the oracle's fused chains, also
where intermediate values are subnormal, infinite or NaN; runs of one, two and more entries, padded strides, inputs
that are only element-aligned."""
import numpy as np
import pytest

import oracle
from helpers import shift_odd_inputs
from kronmult993_amd import workloads as W
from kronmult993_amd.device import DeviceBatch

pytestmark = pytest.mark.gpu

PLANS = [(4, 4), (5, 4), (6, 4), (3, 8), (4, 8)]


def _own_outputs(b):
    return W.HostBatch(**{**b.__dict__, "out_count": b.nb, "out_index": np.arange(b.nb, dtype=np.int64), "out_init": None})


def _check(b, gpu):
    db = DeviceBatch(b, device=str(gpu))
    db.run()
    assert np.array_equal(db.output(), oracle.kronmult(b), equal_nan=True)


@pytest.mark.parametrize("d,n", PLANS)
def test_runs(gpu, d, n):
    for nb in (1, 3, 2051 if n ** d > 600 else 4099):
        b = W.random_case(410 + 7 * d + n, d, n, nb, stride=n + d % 3, shared_factors=37, distinct=nb // 3 + 1,
                          dtype=np.float32)
        _check(shift_odd_inputs(_own_outputs(b)), gpu)


@pytest.mark.parametrize("d,n", PLANS)
def test_subnormal_and_special_values(gpu, d, n):
    """The first contracted factor scales the values into the subnormal range, the last one out of it."""
    b = _own_outputs(W.random_case(430 + 7 * d + n, d, n, 40, dtype=np.float32))
    mats = b.mat_pool.copy()
    for k in range(b.nb):
        for mode, scale in ((d - 1, 1e-10), (0, 1e10)):
            o = int(b.mat_off[k * d + mode])
            mats[o: o + b.stride * n] *= np.float32(scale)
    x = (b.in_pool * np.float32(1e-30)).astype(np.float32)
    x[int(b.in_off[7]) + 5] = np.inf
    x[int(b.in_off[9]) + 3] = np.nan
    _check(W.HostBatch(**{**b.__dict__, "mat_pool": mats, "in_pool": x}), gpu)

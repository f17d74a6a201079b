"""FP32 sweeps of n = 4 and 8 on the matrix cores, factors held in the lanes: bit for bit the oracle's fused chains, also
where intermediate values are subnormal, infinite or NaN; runs of one, two and more entries, padded strides, inputs
that are only element-aligned."""
import numpy as np
import pytest

import oracle
from helpers import accumulation_bound, shift_odd_inputs, terms_reference
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


@pytest.mark.parametrize("d,n", [(3, 9), (3, 10), (4, 6), (4, 7), (4, 9), (4, 10), (5, 5)])
def test_whole_entries(gpu, d, n):
    """n not a multiple of four: the block sweep's rows past n, runs of one, two and more entries, special values."""
    for nb in (1, 3, 1301):
        b = W.random_case(470 + 7 * d + n, d, n, nb, stride=n + d % 3, shared_factors=23, distinct=nb // 3 + 1,
                          dtype=np.float32)
        _check(shift_odd_inputs(_own_outputs(b)), gpu)
    b = _own_outputs(W.random_case(480 + 7 * d + n, d, n, 7, dtype=np.float32))
    x = (b.in_pool * np.float32(1e-39)).astype(np.float32)
    x[int(b.in_off[3]) + 5] = np.inf
    x[int(b.in_off[5]) + 3] = np.nan
    _check(W.HostBatch(**{**b.__dict__, "in_pool": x}), gpu)


@pytest.mark.parametrize("nb,terms", [(1, 2), (5, 1), (700, 1), (2047, 3), (2050, 2), (6147, 2)])
def test_wavefront_per_entry(gpu, nb, terms):
    """d=6 n=4: wavefronts with one entry, several and none; outputs that end inside a wavefront's run, with it, and
    with a workgroup's, so that neighbours' sums are added in every combination."""
    b = W.random_terms(450 + nb, 6, 4, nb, terms, stride=5, shared_factors=29, distinct=nb // 3 + 1, dtype=np.float32)

    def run(c):
        db = DeviceBatch(c, device=str(gpu))
        db.run_terms() if terms > 1 else db.run()
        return db.output()

    own = np.tile(np.arange(nb, dtype=np.int64), terms)
    u = shift_odd_inputs(W.HostBatch(**{**b.__dict__, "out_count": nb, "out_index": own, "out_init": None}))
    assert np.array_equal(run(u), terms_reference(u, True))
    for group in (1, 2, 3, 5, 16):  # consecutive entries per output
        shared = np.tile(np.arange(nb, dtype=np.int64) // group, terms)
        c = W.HostBatch(**{**b.__dict__, "out_count": (nb + group - 1) // group, "out_index": shared, "out_init": None})
        err = np.abs(run(c).astype(np.float64) - oracle.kronmult(c).astype(np.float64))
        assert float(np.max(err - accumulation_bound(c, np.finfo(np.float32).eps / 2))) <= 0.0, group

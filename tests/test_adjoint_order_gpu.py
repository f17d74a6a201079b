"""The adjoint kernels' walk of the entries by input (batches listed by output, a last row that is not full, inputs that
repeat without a period) and their handling of inputs at element-aligned addresses, against the oracle adjoint.
Tolerances as in test_adjoint_gpu.py: only the order of sums differs."""
import numpy as np
import pytest

import oracle
from helpers import normwise
from kronmult993_amd import workloads as W
from kronmult993_amd.device import DeviceBatch

pytestmark = pytest.mark.gpu

TOL = {np.dtype(np.float64): 1e-12, np.dtype(np.float32): 1e-4}


def _batch(seed, d, n, nb, inputs, sets, rows, dtype, gap=0):
    """nb entries: input k % inputs (at a pitch of n^d + gap elements), factor set k % sets, output k // rows."""
    rng = np.random.default_rng(seed)
    size, k = n ** d, np.arange(nb)
    inputs = np.asarray(inputs) if np.ndim(inputs) else k % inputs
    stride = n + 1
    nout = (nb + rows - 1) // rows
    moff = ((k % sets)[:, None] * d + np.arange(d)[None, :]) * (n * stride)
    return W.HostBatch(f"adj_d{d}n{n}_{nb}", d, n, stride, rng.standard_normal(sets * d * n * stride), moff.reshape(-1),
                       rng.standard_normal((int(inputs.max()) + 1) * (size + gap)), inputs * (size + gap), nout, k // rows,
                       grad_out_pool=rng.standard_normal(nout * size)).astype(dtype)


def _check(b, gpu, want_input=True, want_mats=True):
    print(f"[adjoint] {b.name} {b.dtype}", flush=True)
    db = DeviceBatch(b, device=str(gpu))
    db.adjoint_setup(want_input=want_input, want_mats=want_mats)
    db.run_adjoint()
    for got, ref in zip(db.gradients(), oracle.adjoint(b.astype(np.float64), want_input=want_input, want_mats=want_mats)):
        if got is not None:
            assert normwise(got.astype(np.float64), ref) <= TOL[b.dtype]


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("nb,inputs,gap", [(1300, 16, 0), (1297, 18, 1), (1100, 1100, 1), (1100, 1, 0)])
def test_two_modes_per_phase_walks(gpu, nb, inputs, gap, dtype):
    _check(_batch(500 + inputs, 6, 4, nb, inputs, 3, inputs if inputs < nb else 4, dtype, gap), gpu)


def test_inputs_without_a_period(gpu):
    rng = np.random.default_rng(7)
    _check(_batch(510, 6, 4, 1200, rng.integers(0, 37, 1200), 5, 16, np.float64), gpu)


BLOCK_SHAPES = [(3, 5), (3, 6), (3, 7), (4, 3), (4, 5), (4, 6), (4, 7), (4, 8), (5, 3), (5, 4), (5, 5), (6, 2), (6, 3)]


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("d,n", BLOCK_SHAPES)
def test_block_adjoint(gpu, d, n, dtype):
    """Few entries; a batch listed by output with runs of several entries per workgroup and a last row that is not full
    (shared factors: the smaller grid); inputs of their own with factors that take turns; one gradient only."""
    _check(_batch(520 + 9 * d + n, d, n, 5, 5, 2, 2, dtype, 1), gpu)
    nb = 2600 if n ** d <= 700 else 1100
    _check(_batch(530 + 9 * d + n, d, n, nb - 3, 13, 1, 13, dtype, n % 2), gpu)
    _check(_batch(540 + 9 * d + n, d, n, nb + 1, nb + 1, 19, 4, dtype), gpu)
    b = _batch(550 + 9 * d + n, d, n, 90, 7, 5, 6, dtype)
    _check(b, gpu, want_mats=False)
    _check(b, gpu, want_input=False)

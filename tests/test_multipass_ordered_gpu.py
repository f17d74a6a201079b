"""The general multi-pass sweep on d=5 and 6, which unordered calls no longer reach: ordered calls, bit for bit the
documented order of sums over the oracle's contributions."""
import numpy as np
import pytest

from helpers import grouped_by_output, ordered_reference, shift_odd_inputs
from kronmult993_amd import api, workloads as W
from kronmult993_amd.device import DeviceBatch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("d,n,nb,dtype", [(6, 8, 3, np.float32), (6, 6, 4, np.float64), (5, 8, 5, np.float64),
                                          (5, 8, 5, np.float32), (5, 7, 6, np.float64), (6, 5, 5, np.float64),
                                          (5, 9, 4, np.float64), (6, 5, 5, np.float32), (5, 6, 5, np.float64)])
def test_ordered(gpu, d, n, nb, dtype):
    b = shift_odd_inputs(grouped_by_output(W.random_case(730 + 7 * d + n, d, n, nb, distinct=2, dtype=dtype)))
    print(f"[case] ordered d={d} n={n} {b.dtype}", flush=True)
    db = DeviceBatch(b, device=str(gpu), workspace="per_entry")
    db.run_ordered()
    epw = api.ordered_launch_info(d, n, b.dtype.itemsize, nb)["entries_per_workgroup"]
    assert np.array_equal(db.output(), ordered_reference(b, epw))

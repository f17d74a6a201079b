"""The input gradient alone does not pay for the factor gradients' registers: the default kernel takes no longer than the
general one ("recompute"), which keeps everything in LDS (device times of graph replays)."""
import numpy as np
import pytest

from test_walk_cost_gpu import _input_gradient_us

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("d,n,nb,dtype", [(5, 5, 300, np.float64), (5, 5, 1100, np.float64), (4, 7, 520, np.float32),
                                          (4, 7, 700, np.float32), (4, 6, 520, np.float64)])
def test_not_slower_than_the_general_kernel(gpu, d, n, nb, dtype):
    """1.15: the spread of these times from run to run is below a tenth."""
    auto, general = (_input_gradient_us(d, n, nb, nb, dtype, how) for how in ("auto", "recompute"))
    assert auto < 1.15 * general

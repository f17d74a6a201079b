"""Few entries with several terms, d=6 n=4: the FP32 call is not slower than the FP64 one, which moves twice the bytes
through the same steps (device times of graph replays)."""
import numpy as np
import pytest
import torch

from kronmult993_amd import workloads as W
from kronmult993_amd.device import DeviceBatch

pytestmark = pytest.mark.gpu


def _us(nb, terms, dtype):
    b = W.random_terms(460 + nb, 6, 4, nb, terms, stride=4, shared_factors=16, distinct=nb, dtype=dtype)
    db = DeviceBatch(b)
    s = torch.cuda.Stream()
    with torch.cuda.stream(s):
        db.run_terms(sync=False, stream=s)
        s.synchronize()
        g = torch.cuda.CUDAGraph()
        with torch.cuda.graph(g, stream=s):
            for _ in range(10):
                db.run_terms(sync=False, stream=s)
        times = []
        for _ in range(7):
            a, e = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            a.record(s)
            g.replay()
            e.record(s)
            e.synchronize()
            times.append(a.elapsed_time(e) * 100)
    print(f"[terms] {nb} x {terms} {np.dtype(dtype).name}: {min(times):.2f} us", flush=True)
    return min(times)


@pytest.mark.parametrize("nb,terms", [(16, 3), (16, 5), (100, 3), (100, 5)])
def test_few_entries(gpu, nb, terms):
    """1.05: the spread of these times from run to run."""
    assert _us(nb, terms, np.float32) < 1.05 * _us(nb, terms, np.float64)

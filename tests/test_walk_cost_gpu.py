"""What the adjoint's walk of the entries by input costs and gives (device times of graph replays; the ratios leave a
factor of 1.4 and more to what is expected)."""
import numpy as np
import pytest
import torch

from kronmult993_amd import workloads as W
from kronmult993_amd.device import DeviceBatch

pytestmark = pytest.mark.gpu


def _input_gradient_us(d, n, nb, inputs, dtype, intermediates="auto"):
    """Fastest of seven replays of ten calls: entry k has input k % inputs."""
    size, k = n ** d, np.arange(nb)
    rng = np.random.default_rng(nb + inputs)
    x, m = rng.standard_normal(inputs * size), rng.standard_normal(16 * d * n * n)
    off = ((k % 16)[:, None] * d + np.arange(d)[None, :]) * (n * n)
    b = W.HostBatch(f"walk_d{d}n{n}_{nb}_{inputs}", d, n, n, m, off.reshape(-1), x, (k % inputs) * size, nb // 4 + 1,
                    k // 4, grad_out_pool=rng.standard_normal((nb // 4 + 1) * size)).astype(dtype)
    db = DeviceBatch(b)
    db.adjoint_setup(want_mats=False, intermediates=intermediates)
    s = torch.cuda.Stream()
    with torch.cuda.stream(s):
        db.run_adjoint(sync=False, stream=s)
        s.synchronize()
        g = torch.cuda.CUDAGraph()
        with torch.cuda.graph(g, stream=s):
            for _ in range(10):
                db.run_adjoint(sync=False, stream=s)
        times = []
        for _ in range(7):
            a, e = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            a.record(s)
            g.replay()
            e.record(s)
            e.synchronize()
            times.append(a.elapsed_time(e) * 100)
    print(f"[walk] {b.name} {b.dtype}: {min(times):.2f} us", flush=True)
    return min(times)


@pytest.mark.parametrize("d,n,dtype", [(6, 2, np.float64), (3, 5, np.float32), (3, 7, np.float32)])
def test_looking_for_the_period_is_cheap(gpu, d, n, dtype):
    """Where a batch outgrows the resident workgroups they look for the period first. Half as many entries again cost
    at most half the time again, a second round of entries and one trip to memory: below 2.2 times in all (a search
    that is a chain of loads: 2.5 to 3.2 times)."""
    sizes = (1400, 2100, 3100, 4400, 6300, 9400, 14000, 20000)
    t = [_input_gradient_us(d, n, nb, nb, dtype) for nb in sizes]
    assert max(b / a for a, b in zip(t, t[1:])) < 2.2, t


@pytest.mark.parametrize("period", [5, 64, 1000])
def test_a_period_is_found(gpu, period):
    """8192 entries, at least 8 to an input: an eighth of the input gradients' atomic adds, most of the time without."""
    assert _input_gradient_us(6, 4, 8192, period, np.float64) < 0.7 * _input_gradient_us(6, 4, 8192, 8192, np.float64)

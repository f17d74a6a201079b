"""GPU parity of the block sweep (whole entries in LDS, and the block pass plus the register pass of larger vectors)
with the oracle: bit for bit where each output has one contribution, within the accumulation bound where outputs are
shared. Runs are cut inside and between outputs, strides are padded and odd entries' inputs only element-aligned."""
import numpy as np
import pytest

import oracle
from helpers import accumulation_bound, grouped_by_output, normwise, shift_odd_inputs
from kronmult993_amd import api, workloads as W
from kronmult993_amd.device import DeviceBatch

pytestmark = pytest.mark.gpu

DTYPES = [np.float64, np.float32]
EPS = {np.dtype(np.float64): np.finfo(np.float64).eps / 2, np.dtype(np.float32): np.finfo(np.float32).eps / 2}


def _run(b, gpu):
    print(f"[case] {b.name} d={b.d} n={b.n} nb={b.nb} {b.dtype}", flush=True)
    db = DeviceBatch(b, device=str(gpu), workspace="per_entry")
    inputs = db.inp.clone()
    db.run()
    assert bool((db.inp == inputs).all())
    return db.output()


def _check(b, gpu):
    u = W.HostBatch(**{**b.__dict__, "out_count": b.nb, "out_index": np.arange(b.nb, dtype=np.int64), "out_init": None})
    assert np.array_equal(_run(u, gpu), oracle.kronmult(u))
    for case in (b, grouped_by_output(b)):
        err = np.abs(_run(case, gpu).astype(np.float64) - oracle.kronmult(case).astype(np.float64))
        assert float(np.max(err - accumulation_bound(case, EPS[case.dtype]))) <= 0.0


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("d,n", [(3, 6), (3, 7), (3, 9), (3, 10), (4, 5), (4, 6), (4, 7), (4, 9), (4, 10), (5, 5),
                                 (5, 6), (6, 3), (6, 5)])
def test_whole_entries(gpu, d, n, dtype):
    assert api.kernel_name(d, n, np.dtype(dtype).itemsize, 50).startswith(("fiber", "wave", "multipass"))
    _check(shift_odd_inputs(W.random_case(310 + 7 * d + n, d, n, 50, stride=n + d % 3, shared_factors=17, dtype=dtype)),
           gpu)


@pytest.mark.parametrize("d,n,dtype,nb", [(3, 6, np.float64, 2600), (4, 5, np.float64, 1700), (4, 7, np.float32, 1300),
                                          (5, 5, np.float64, 1100), (4, 9, np.float64, 600), (6, 3, np.float32, 2500)])
def test_runs_of_entries(gpu, d, n, dtype, nb):
    """More entries than resident workgroups: runs of two and more entries, a shorter last one."""
    _check(W.random_case(330 + d + n, d, n, nb, stride=n + 1, shared_factors=211, distinct=nb // 4 + 1, dtype=dtype), gpu)


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("d,n", [(5, 7), (5, 8), (5, 9), (5, 10), (6, 5), (6, 6), (6, 7), (6, 8), (6, 9), (6, 10)])
def test_large_vectors(gpu, d, n, dtype):
    """Two passes; 9 entries of 3 outputs leave the four wavefronts of a workgroup on one output or on several."""
    nb = 9 if n ** d <= 300000 else 5
    _check(shift_odd_inputs(W.random_case(350 + 7 * d + n, d, n, nb, stride=n + n % 3, shared_factors=3, distinct=3,
                                          dtype=dtype)), gpu)


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("d,n", [(4, 3), (5, 3), (7, 2), (8, 2), (3, 6), (3, 7), (4, 5)])
def test_whole_fibers_per_lane(gpu, d, n, dtype):
    """One wavefront per entry: fewer entries than a workgroup's wavefronts, one per wavefront and two, the last
    workgroup partly without entries; wavefronts of a workgroup on one output and on several."""
    for nb in (3, 101, 4403):
        _check(shift_odd_inputs(W.random_case(360 + 7 * d + n, d, n, nb, stride=n + d % 3, shared_factors=57,
                                              distinct=nb // 6 + 1, dtype=dtype)), gpu)


@pytest.mark.parametrize("family", [api.FAMILY_WAVE, api.FAMILY_FIBER, api.FAMILY_PACKED])
def test_whole_fibers_per_lane_families(gpu, family):
    """d=3 n=6 through each family that it belongs to, with run lengths and grids asked for."""
    b = W.random_case(377, 3, 6, 333, distinct=40)
    u = W.HostBatch(**{**b.__dict__, "out_count": b.nb, "out_index": np.arange(b.nb, dtype=np.int64), "out_init": None})
    ref = oracle.kronmult(u)
    for epw, wpc in ((0, 0), (1, 0), (7, 0), (2000000000, 0), (0, 1)):
        tu = {"family": family, "entries_per_workgroup": epw, "workgroups_per_cu": wpc}
        if family == api.FAMILY_PACKED and epw > 1000:
            continue
        db = DeviceBatch(u, device=str(gpu))
        db.run(tuning=tu)
        assert np.array_equal(db.output(), ref), tu


def test_large_vectors_run_lengths(gpu):
    """Enough entries for runs of several per wavefront and of several blocks per workgroup (d=5 n=9 and d=5 n=7)."""
    _check(W.random_case(371, 5, 7, 1500, shared_factors=40, distinct=7, dtype=np.float32), gpu)
    _check(W.random_case(372, 5, 9, 300, shared_factors=40, distinct=5, dtype=np.float64), gpu)


@pytest.mark.parametrize("d,n,dtype,nb", [(5, 8, np.float64, 1026), (5, 8, np.float32, 1030), (5, 10, np.float32, 515),
                                          (5, 7, np.float64, 1029), (5, 10, np.float64, 513)])
def test_large_vectors_long_runs(gpu, d, n, dtype, nb):
    """Runs of four entries and more: row blocks that share a workgroup, reads past the caches; a last workgroup with
    a short part or without its second one."""
    _check(shift_odd_inputs(W.random_case(390 + n, d, n, nb, stride=n + n % 3, shared_factors=41, distinct=5,
                                          dtype=dtype)), gpu)


@pytest.mark.parametrize("d,n,itemsize", [(4, 10, 8), (5, 7, 8), (6, 5, 8), (6, 10, 4)])
def test_large_vectors_need_a_workspace(gpu, d, n, itemsize):
    dtype = np.float64 if itemsize == 8 else np.float32
    assert api.launch_info(d, n, itemsize, 2)["uses_workspace"] == 1
    db = DeviceBatch(W.random_case(380, d, n, 2, dtype=dtype), device=str(gpu), workspace="none")
    with pytest.raises(api.KronmultError):
        db.run()


@pytest.mark.parametrize("strategy", ["auto", "persistent"])
@pytest.mark.parametrize("dtype", DTYPES)
def test_grouped_paths(gpu, dtype, strategy):
    """Every path of the grouped launch, tables with and without passes, default tiles and tiles that leave wavefronts
    without entries; a group large enough for a launch of its own under "auto" (d=5 n=4)."""
    import torch
    small = [(3, 5, 37), (3, 6, 90), (4, 3, 61), (4, 4, 45), (5, 3, 33), (7, 2, 18), (8, 2, 19), (2, 8, 70), (6, 2, 9)]
    for shapes in (small, small[:2] + [(3, 7, 40), (4, 5, 21), (5, 4, 1100)]):
        for tile in (0, 1, 6, 31):
            bs = [W.random_case(390 + 10 * d + n, d, n, nb, stride=n + 1, distinct=nb, dtype=dtype) for d, n, nb in shapes]
            bs = [W.HostBatch(**{**b.__dict__, "out_init": np.zeros_like(b.out_init)}) for b in bs]
            dbs = [DeviceBatch(b, device=str(gpu)) for b in bs]
            print(f"[grouped] {strategy} tile={tile} {shapes}", flush=True)
            api.kronmult_batched_grouped([db.group(entries_per_tile=tile) for db in dbs], dtype=dbs[0].dtype_name,
                                         strategy=strategy)
            torch.cuda.synchronize()
            for b, db in zip(bs, dbs):
                assert np.array_equal(db.output(), oracle.kronmult(b)), (b.d, b.n, tile)


def test_grouped_shared_outputs(gpu):
    import torch
    bs = [W.random_case(410 + d, d, n, nb, distinct=nb // 5) for d, n, nb in ((3, 6, 300), (5, 3, 211), (4, 4, 97))]
    bs = bs + [grouped_by_output(b) for b in bs]
    dbs = [DeviceBatch(b, device=str(gpu)) for b in bs]
    api.kronmult_batched_grouped([db.group() for db in dbs], dtype="f64")
    torch.cuda.synchronize()
    for b, db in zip(bs, dbs):
        assert float(np.max(np.abs(db.output() - oracle.kronmult(b)) - accumulation_bound(b, EPS[b.dtype]))) <= 0.0

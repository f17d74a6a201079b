"""Hints of a grouped call's large groups under "auto": they are followed as in the persistent strategy, and a tuning that
only a launch of its own reads does not make the call fail."""
import numpy as np
import pytest
import torch

import oracle
from kronmult993_amd import api, workloads as W
from kronmult993_amd.device import DeviceBatch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("tile,wpc", [(0, 0), (16, 0), (0, 4), (3, 2)])
@pytest.mark.parametrize("tuning", [None, {"family": api.FAMILY_WAVE}, {"family": api.FAMILY_MATRIX},
                                    {"entries_per_workgroup": 5}])
def test_auto_keeps_large_groups_with_hints(gpu, tile, wpc, tuning):
    """d=5 n=4, 1100 entries: above 2^20 elements; the wave and matrix families do not cover the shape."""
    bs = [W.random_case(720, 5, 4, 1100, distinct=1100), W.random_case(721, 3, 4, 50, distinct=50)]
    bs = [W.HostBatch(**{**b.__dict__, "out_init": np.zeros_like(b.out_init)}) for b in bs]
    dbs = [DeviceBatch(b, device=str(gpu)) for b in bs]
    print(f"[grouped] auto tile={tile} wpc={wpc} tuning={tuning}", flush=True)
    groups = [dbs[0].group(tuning=tuning, entries_per_tile=tile), dbs[1].group()]
    api.kronmult_batched_grouped(groups, dtype="f64", strategy="auto", workgroups_per_cu=wpc)
    torch.cuda.synchronize()
    for b, db in zip(bs, dbs):
        assert np.array_equal(db.output(), oracle.kronmult(b))


def test_separate_still_refuses_a_tuning_that_does_not_cover_the_shape(gpu):
    db = DeviceBatch(W.random_case(722, 5, 4, 1100), device=str(gpu))
    with pytest.raises(api.KronmultError):
        api.kronmult_batched_grouped([db.group(tuning={"family": api.FAMILY_WAVE})], dtype="f64", strategy="separate")

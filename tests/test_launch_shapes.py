"""The launch that a tuning asks for is the one that is made (launch_info; no device needed)."""
import pytest

from kronmult993_amd import api

WHOLE_FIBERS = [(4, 3), (5, 3), (7, 2), (8, 2), (3, 6)]


@pytest.mark.parametrize("itemsize", [8, 4])
@pytest.mark.parametrize("d,n", WHOLE_FIBERS + [(3, 4), (3, 5), (2, 9)])
def test_wave_family_entries_per_workgroup(d, n, itemsize):
    for nb in (1, 333, 20000):
        for epw in (1, 2, 5, 7, 8, 64, nb + 3):
            info = api.launch_info(d, n, itemsize, nb, {"family": api.FAMILY_WAVE, "entries_per_workgroup": epw})
            assert info["entries_per_workgroup"] == epw
            assert info["grid"] == (-(-nb // epw) + 7) // 8 * 8


@pytest.mark.parametrize("d,n", WHOLE_FIBERS)
def test_wave_family_workgroups_per_cu(d, n):
    """The run and the grid of the family's one-element shapes."""
    for nb, wpc in ((20000, 1), (20000, 7), (300, 2), (5000, 16)):
        tu = {"family": api.FAMILY_WAVE, "workgroups_per_cu": wpc}
        info, one = api.launch_info(d, n, 8, nb, tu), api.launch_info(3, 4, 8, nb, tu)
        assert (info["entries_per_workgroup"], info["grid"]) == (one["entries_per_workgroup"], one["grid"])

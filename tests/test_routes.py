"""Which kernel a shape runs on, by its name and its launch shape (no device needed: launch information is computed on
the host), so that a shape that falls back to a general kernel of the same results is noticed."""
import pytest

from kronmult993_amd import api

BLOCK = [(3, 9), (3, 10), (4, 6), (4, 7), (4, 9), (4, 10), (5, 5), (5, 6), (6, 3)]
PASS_THREADS = {5: (64, 64), 6: (128, 64), 7: (192, 128), 8: (512, 256), 9: (768, 768), 10: (1024, 512)}  # FP64, FP32


def _sfx(itemsize):
    return "f64" if itemsize == 8 else "f32"


@pytest.mark.parametrize("d,n,itemsize", [(d, n, i) for d, n in BLOCK for i in (8, 4)] + [(6, 5, 4)])
def test_block_sweep(d, n, itemsize):
    """One thread per fiber, as few per thread as 1024 threads leave; the whole vector in LDS (rows of 8 padded)."""
    assert api.kernel_name(d, n, itemsize, 50) == \
        ("fiber_global" if n ** d * itemsize > 65000 else "fiber_lds") + "_block_" + _sfx(itemsize)
    info = api.launch_info(d, n, itemsize, 4608)
    fibers = n ** (d - 1)
    per = -(-fibers // 1024)
    assert info["family"] == api.FAMILY_FIBER
    assert info["block"] == (-(-fibers // per) + 63) // 64 * 64 and info["lds_bytes"] == n ** d * itemsize
    assert info["entries_per_workgroup"] > 1  # runs (the general kernel: one workgroup per entry)


@pytest.mark.parametrize("itemsize", [8, 4])
@pytest.mark.parametrize("d,n", [(5, 7), (5, 8), (5, 9), (5, 10), (6, 5), (6, 6), (6, 7), (6, 8), (6, 9), (6, 10)])
def test_two_passes(d, n, itemsize):
    """The block pass over n^4 elements a block; an ordered call of the same shape keeps the general kernel."""
    if (d, n, itemsize) == (6, 5, 4):
        return
    assert api.kernel_name(d, n, itemsize, 50) == "multipass_" + _sfx(itemsize)
    info, general = api.launch_info(d, n, itemsize, 50), api.ordered_launch_info(d, n, itemsize, 50)
    assert info["uses_workspace"] == 1 and info["block"] == PASS_THREADS[n][0 if itemsize == 8 else 1]
    pad = n ** 3 * 16 if n == 8 else 0
    assert info["lds_bytes"] == n ** 4 * itemsize + pad
    assert (info["block"], info["lds_bytes"]) != (general["block"], general["lds_bytes"])


@pytest.mark.parametrize("itemsize", [8, 4])
@pytest.mark.parametrize("d,n", [(7, 5), (8, 4), (9, 3), (15, 3)])
def test_general_passes(d, n, itemsize):
    """Shapes that the two-pass kernels are not built for."""
    if n ** d * itemsize <= 64 * 1024:
        return
    assert api.kernel_name(d, n, itemsize, 2) == "multipass_" + _sfx(itemsize)
    info, general = api.launch_info(d, n, itemsize, 2), api.ordered_launch_info(d, n, itemsize, 2)
    assert (info["block"], info["lds_bytes"]) == (general["block"], general["lds_bytes"])


@pytest.mark.parametrize("itemsize", [8, 4])
@pytest.mark.parametrize("d,n", [(4, 3), (5, 3), (7, 2), (8, 2), (3, 6), (3, 7), (4, 5)])
def test_whole_fibers_per_lane(d, n, itemsize):
    """Four wavefronts per workgroup, one or two entries each, whatever family the shape belongs to by default."""
    for nb, epw in ((50, 4), (20000, 8)):
        info = api.launch_info(d, n, itemsize, nb)
        assert (info["block"], info["entries_per_workgroup"]) == (256, epw)
    if (d, n) in ((3, 7), (4, 5)):
        assert api.kernel_name(d, n, itemsize, 50) == "fiber_lds_wave_" + _sfx(itemsize)


def test_wavefront_per_entry_d6n4():
    info = api.launch_info(6, 4, 4, 700)
    assert (info["entries_per_workgroup"], info["lds_bytes"]) == (4, 4 * 4096 * 4)
    assert api.kernel_name(6, 4, 4, 700) == "reg_sweep_wave_f32"
    for nb in (100, 8192):
        assert api.kernel_name(6, 4, 4, nb) == "reg_sweep_f32" and api.launch_info(6, 4, 4, nb)["lds_bytes"] == 4096 * 4
    assert api.ordered_launch_info(6, 4, 4, 700)["lds_bytes"] == 4096 * 4

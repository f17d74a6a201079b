"""What an untuned call runs is among the autotuner's candidates, so that a tuned call is not slower (no device: the
timing is replaced)."""
import pytest

from kronmult993_amd import api, autotune


class Batch:
    device, dtype_name = "none", "f32"

    def __init__(self, d, n, nb, itemsize=4):
        self.d, self.n, self.nb, self.itemsize, self.size = d, n, nb, itemsize, n ** d
        self.calls = []

    def run(self, sync, tuning, stream):
        self.calls.append(dict(tuning))

    def group(self, tuning=None, entries_per_tile=0):
        return tuning, entries_per_tile


@pytest.fixture
def tuner(monkeypatch):
    monkeypatch.setattr(autotune, "arch", lambda device: "test")
    monkeypatch.setattr(autotune, "_CACHE", {})
    monkeypatch.delenv("KRONMULT_TUNE_CACHE", raising=False)
    return autotune.Autotuner()


def _default(tuning):
    return not any(tuning.get(k, 0) for k in ("family", "workgroups_per_cu", "entries_per_workgroup"))


@pytest.mark.parametrize("d,n,nb", [(6, 4, 1000), (3, 6, 5000), (5, 5, 300)])
def test_single(tuner, monkeypatch, d, n, nb):
    """The default is timed, and kept when it is the fastest; its choice can be passed on as a tuning."""
    db = Batch(d, n, nb)

    def time_us(fn):
        fn(None)
        return 1.0 if _default(db.calls[-1]) else 2.0

    monkeypatch.setattr(tuner, "_time_us", time_us)
    choice = tuner.tune_single(db)
    assert any(_default(c) for c in db.calls) and _default(choice)
    assert api.launch_info(d, n, 4, nb, {k: v for k, v in choice.items() if k != "us"}) == api.launch_info(d, n, 4, nb)


@pytest.mark.parametrize("shapes,fastest", [([(5, 4, 3000), (2, 8, 6000)], "auto"),
                                            ([(3, 6, 900), (2, 8, 700)], "persistent")])
def test_grouped(tuner, monkeypatch, shapes, fastest):
    """Large groups: the automatic strategy is timed; the persistent launch in its default shape always is."""
    calls = []

    def grouped(groups, *, dtype, strategy, workgroups_per_cu=0, stream=None, structs=None):
        calls.append((strategy, workgroups_per_cu, [tile for _, tile in groups]))

    def time_us(fn):
        before = len(calls)
        fn(None)
        return 1.0 if len(calls) > before and calls[-1] == (fastest, 0, [0] * len(shapes)) else 2.0

    monkeypatch.setattr(api, "kronmult_batched_grouped", grouped)
    monkeypatch.setattr(api, "grouped_structs", lambda groups, dtype: None)
    monkeypatch.setattr(tuner, "_time_us", time_us)
    dbs = [Batch(*s) for s in shapes]
    choice = tuner.tune_grouped(dbs)
    assert (choice["strategy"], choice["workgroups_per_cu"], choice["entries_per_tile"]) == (fastest, 0, [0] * len(dbs))
    _, _, kwargs = autotune.grouped_call_from_choice(dbs, choice)
    assert kwargs == {"strategy": fastest, "workgroups_per_cu": 0}

"""The variant cache and slots whose work the whole-run kernel of a 1D problem does: a stored
choice of stage kernels is not applied to them (selecting a stage kernel would switch the run
kernel off), whatever it says.  Host only, on a stand-in object.
"""
import json

import pytest

from passivetracerflows import tuning

from test_tuning_cache import FakeSlots


class RunSlots(FakeSlots):
    def __init__(self, names, variants, run):
        super().__init__(names, variants)
        self.run = run

    def whole_run(self, i):
        return self.run[i]

    def autotune(self):
        self.tuned += 1      # nothing to choose


NAMES = [f"stage{s}_x_advect_stage" for s in (1, 2, 3, 4)]


@pytest.mark.parametrize("stored", [(4, 1), (8, 2)])
def test_stored_choice_leaves_the_run_kernel_on(tmp_path, stored):
    path = str(tmp_path / "tuning.json")
    with open(path, "w") as f:
        json.dump({"key": [[n, *stored, False, False, False] for n in NAMES]}, f)
    obj = RunSlots(NAMES, [(4, 1, False, False, False)] * 4, [True] * 4)
    assert tuning.apply_or_tune(obj, "key", path) == "cache"
    assert obj.set_calls == [] and obj.tuned == 0
    # the stage kernels of a problem that runs them take it
    obj = RunSlots(NAMES, [(4, 1, False, False, False)] * 4, [False] * 4)
    assert tuning.apply_or_tune(obj, "key", path) == "cache"
    assert [c[0] for c in obj.set_calls] == [0, 1, 2, 3]


def test_tuned_then_loaded_is_the_same(tmp_path):
    path = str(tmp_path / "tuning.json")
    for how in ("tuned", "cache"):
        obj = RunSlots(NAMES, [(4, 1, False, False, False)] * 4, [True] * 4)
        assert tuning.apply_or_tune(obj, "key", path) == how
        assert obj.set_calls == []

"""Recorded launch policies of other kernels are not installed."""
import pytest

from staccato_amd import autotune


class Recorder:
    def __init__(self):
        self.set = []

    def set_policy(self, *a):
        self.set.append(a)


ENTRY = {"name": "register-panel", "kernel": 1, "lds_budget": 0, "jb_max": 0, "pts_per_s": 2.0e6}


@pytest.mark.parametrize("generation", [None, autotune.GENERATION - 1, autotune.GENERATION + 1])
def test_entry_of_another_generation_is_ignored(generation):
    entry = dict(ENTRY) if generation is None else dict(ENTRY, generation=generation)
    h = Recorder()
    assert not autotune.apply_cached(h, 60, 1, "plain", {autotune._key(60, 1, "plain"): entry})
    assert h.set == []


def test_entry_of_this_generation_is_installed():
    h = Recorder()
    cache = {autotune._key(60, 1, "plain"): dict(ENTRY, generation=autotune.GENERATION)}
    assert autotune.apply_cached(h, 60, 1, "plain", cache)
    assert h.set == [(60, "plain", 1, 0, 0)]

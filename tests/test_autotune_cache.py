"""The autotuner's cache and choices on a level that only counts (no GPU): a
choice is reused for the same boxes, one timed with another launch structure
is not, and the first-flux faces get the settings they take."""
import json

import pytest

from camr_amd import _lib, autotune, workloads


class CountingLevel:
    """Level's tuning interface; every stage takes 1 ms, 0.5 ms in blocks of
    64, and the whole step the stages' sum."""

    def __init__(self):
        self.prob = workloads.smooth_periodic(n=16)
        self.runs = 0
        self._profile = False
        self.xcd, self.ctu = [16] * _lib.NSTAGE, (0, 8)
        self.tuning = ([256] * _lib.NSTAGE, 0)

    @property
    def tuning(self):
        return self._blocks, self._order

    @tuning.setter
    def tuning(self, t):
        self._blocks, self._order = list(t[0]), t[1]
        self.tiles = [autotune.LINEAR] * _lib.NSTAGE

    def run(self, steps):
        self.runs += steps

    def sync(self):
        pass

    def profile(self, on):
        self._profile = on

    def profile_report(self):
        return {n: {"ms": 0.5 if self._blocks[st[0]] == 64 else 1.0, "count": 1}
                for n, st in autotune.STAGES.items()}


@pytest.fixture
def cache(tmp_path, monkeypatch):
    path = tmp_path / "tuning.json"
    monkeypatch.setenv("CAMR_TUNING_CACHE", str(path))
    monkeypatch.setattr(autotune, "_device_name", lambda: "dev")
    # the tuned shapes always win the whole-step check
    times = iter(range(1, 1000))
    monkeypatch.setattr(autotune, "_step_time", lambda level, steps: float(next(times)))
    return path


def test_choice_is_reused_for_the_same_launches(cache):
    first = CountingLevel()
    got = autotune.tune(first, steps=1)
    assert first.runs > 0
    again = CountingLevel()
    assert autotune.tune(again, steps=1) == got and again.runs == 0
    assert again.tuning == first.tuning


def test_choice_of_other_launches_is_not_applied(cache):
    level = CountingLevel()
    key = autotune.key_of(level, "dev")
    old = [64 if k % 2 else 128 for k in range(_lib.NSTAGE)]  # keeps every stage apart
    entry = {"blocks": old, "order": 1, "tiles": [[0, 0, 0]] * _lib.NSTAGE,
             "xcd": [0] * _lib.NSTAGE, "ctu": [0, 8]}
    other = key.replace(f"launches{autotune.LAUNCHES}|", "")
    assert other != key
    cache.write_text(json.dumps({other: entry}))
    blocks = autotune.tune(level, steps=1)[0]
    assert level.runs > 0 and blocks != old
    for grp in autotune.GROUPS:
        assert len({blocks[g] for g in grp}) == 1
    kept = json.loads(cache.read_text())
    assert kept[other] == entry and key in kept


def test_first_flux_faces_take_only_the_xcd_chunk(cache):
    blocks, _, tiles, xcd, _ = autotune.tune(CountingLevel(), steps=1)
    for s in range(_lib.NSTAGE):
        face1 = s in (2, 3, 4)
        assert blocks[s] == (256 if face1 else 64)
        assert not face1 or tiles[s] == autotune.LINEAR
    assert xcd[2] in autotune.XCD_CHUNKS
    assert [c[2] for c in autotune.candidates((2, 3, 4))] == list(autotune.XCD_CHUNKS)

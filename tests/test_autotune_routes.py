"""The tuner on batches whose plan takes two launches, which heed the pixels per
lane and culling only (host logic, with a clock of its own)."""
import torch

from forcepho_amd import autotune


class Batch:
    """Two launches up to 4 pixels per lane; times by pixels per lane there, and
    by workgroups per CU too with one wave per tile."""

    def __init__(self, limit):
        self.limit, self.launches = limit, []

    def set_launch(self, **launch):
        self.launch = launch
        self.launches.append(launch)

    def two_launches(self):
        return self.launch["pix_per_lane"] <= self.limit

    def ms(self):
        K = self.launch["pix_per_lane"]
        if self.two_launches():
            # noise that differs from call to call, beyond the tie
            return 10.0 / K + 0.5 * (len(self.launches) % 7)
        return 40.0 / K + 1.0 / self.launch["groups_per_cu"] + self.launch["persistent"]


def tune(monkeypatch, batch):
    class Event:
        def __init__(self, enable_timing):
            pass

        def record(self):
            pass

        def elapsed_time(self, other):
            return 3 * batch.ms()

    monkeypatch.setattr(torch.cuda, "Event", Event)
    monkeypatch.setattr(torch.cuda, "synchronize", lambda: None)
    return autotune.tune(batch, lambda: None)


def test_two_launches_are_timed_once_and_keep_the_knobs_they_do_not_heed(monkeypatch):
    kept = dict(pix_per_lane=2, waves_per_group=3, persistent=1, groups_per_cu=7, cull=1)
    monkeypatch.setattr(autotune, "load_or_default", lambda kind="batch": dict(kept))
    batch = Batch(limit=8)
    best, table = tune(monkeypatch, batch)
    assert sorted(c["pix_per_lane"] for _, c in table) == [1, 2, 4, 8]
    for _, c in table:
        assert c == dict(kept, pix_per_lane=c["pix_per_lane"])
    assert batch.launch == best


def test_one_wave_per_tile_is_timed_at_every_candidate(monkeypatch):
    best, table = tune(monkeypatch, Batch(limit=0))
    assert [c for _, c in table if c["pix_per_lane"] == 8] and len(table) == \
        len(autotune.candidates("batch"))
    assert best["pix_per_lane"] == 8 and best["persistent"] == 0
    _, mixed = tune(monkeypatch, Batch(limit=2))
    assert len(mixed) == len(autotune.candidates("batch")) // 2 + 2

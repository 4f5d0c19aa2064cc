"""The autotuner's choice, with the times given: no GPU."""
import pytest

from bvhtracer_amd import autotune


def tuned(monkeypatch, times, configs=None):
    state = {"set": None}
    monkeypatch.setattr(autotune, "set_config", lambda ctx, wg, d: state.update(set=(wg, d)))
    monkeypatch.setattr(autotune, "time_ms", lambda ctx, run, reps: times.get(state["set"], 9.0))
    best, table = autotune.tune(None, lambda: None, configs=configs)
    assert state["set"] == best
    return best, table


@pytest.mark.parametrize("times,best", [({(0, 0): 0.17, (64, 24): 3.1}, (0, 0)),
                                        ({(0, 0): 1.0, (128, 8): 0.9}, (128, 8)),
                                        ({(0, 0): 1.0, (64, 24): 0.995}, (0, 0))])
def test_the_default_is_a_candidate_and_wins_ties(monkeypatch, times, best):
    got, table = tuned(monkeypatch, times)
    assert got == best
    assert list(table) == [(0, 0)] + autotune.configurations() and len(table) == 13


def test_given_configurations_are_the_only_candidates(monkeypatch):
    got, table = tuned(monkeypatch, {(0, 0): 0.1, (64, 8): 2.0, (256, 8): 1.0}, [(64, 8), (256, 8)])
    assert got == (256, 8) and set(table) == {(64, 8), (256, 8)}

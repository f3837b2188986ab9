"""The tuner leaves out the options that contexts accept without effect: it neither times nor recommends them."""
import numpy as np
import pytest

from disccofan_amd import tune

IMG = np.zeros((4, 4), np.uint8)


@pytest.fixture
def runs(monkeypatch):
    """settings that were run; every run is faster than the one before, as noise may have it"""
    seen = []

    def run(self, setting):
        seen.append(dict(setting))
        return 1.0 / len(seen), [np.zeros(3)]
    monkeypatch.setattr(tune._Runner, "run", run)
    return seen


@pytest.mark.parametrize("img", [IMG, np.zeros((2, 4, 4), np.uint8)])
def test_single_images_run_once(runs, img):
    best, s, table = tune.tune([img], [1.0])
    assert len(runs) == 1 and s == 1.0
    assert best == {k: v[0] for k, v in tune.knobs_for(img.ndim == 3, False).items()}
    assert all(row[1] == 1.0 for row in table)


@pytest.mark.parametrize("grid", [None, (1, 2)])
def test_only_options_with_an_effect_are_run(runs, grid):
    knobs = tune.knobs_for(False, grid is None, grid is not None)
    best, _, table = tune.tune([IMG], [1.0], batched=grid is None, grid=grid)
    live = [k for k in knobs if k not in tune.NO_EFFECT]
    assert live and len(runs) == 1 + sum(len(knobs[k]) - 1 for k in live)
    assert all(best[k] == knobs[k][0] for k in knobs if k in tune.NO_EFFECT)
    assert len(table) == 1 + sum(len(v) - 1 for v in knobs.values())


@pytest.mark.parametrize("workload", ["vnoise", "batch", "tiled"])
def test_cli_recommends_options_with_an_effect(runs, workload, capsys):
    tune.main(["--workload", workload, "--size", "64", "--count", "2", "--lo", "64"])
    out = capsys.readouterr().out.splitlines()
    names = [w.split("=")[0] for w in out[-1].split() if "=" in w]
    assert not set(names) & tune.NO_EFFECT
    assert bool(names) == (workload != "vnoise") and (len(runs) > 1) == (workload != "vnoise")

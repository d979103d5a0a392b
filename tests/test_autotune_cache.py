"""The autotuner's cache file on the CPU: entries are used, unless they were
written before the automatic choice was among the candidates."""
import json

import numpy as np
import pytest

from cemc_amd import autotune


class _Model:
    n_sites, n_species, n_subclusters = 64, 2, 12


class _Batch:
    """Runs twice as fast on the automatic choice."""
    made = 0

    def __init__(self, models, chains):
        type(self).made += 1
        self.n_chains = len(chains)
        self.shape = [0, 0, 0]

    def set_energy_path(self, path):
        self.shape[2] = path

    def set_moves_per_round(self, moves):
        self.shape[1] = moves

    def set_waves(self, waves):
        self.shape[0] = waves

    def energy_path(self, chain):
        return autotune.PATH_EVALUATE

    def launch_shape(self, chain):
        return tuple(self.shape)

    def run(self, moves):
        pass

    def run_timed(self, moves):
        return 1.0 if tuple(self.shape) == autotune.AUTO else 2.0

    def close(self):
        pass


@pytest.mark.parametrize("rates,timed", [
    ({"4x8": 9.0, "1x1": 3.0}, True),
    ({"4x8": 9.0, "1x1": 3.0, "auto": 5.0}, False),
])
def test_entries_without_the_automatic_choice_are_timed_again(monkeypatch, tmp_path, rates, timed):
    models, chains = [_Model()] * 2, [dict(kind=0)] * 2
    sig = autotune.signature(models, chains)
    path = tmp_path / "shapes.json"
    path.write_text(json.dumps({sig: {"best": [4, 8, autotune.PATH_EVALUATE], "rates": rates}}))
    monkeypatch.setattr(autotune, "_cache", {})
    monkeypatch.setattr(autotune, "ChainBatch", _Batch)
    _Batch.made = 0
    best, got = autotune.tune(models, chains, cache_file=str(path))
    assert (_Batch.made == 1) == timed
    assert best == (autotune.AUTO if timed else (4, 8, autotune.PATH_EVALUATE))
    assert autotune.AUTO in got or not timed
    stored = json.loads(path.read_text())[sig]
    assert tuple(stored["best"]) == best and "auto" in stored["rates"]
    assert np.isfinite(list(stored["rates"].values())).all()

"""Wang-Landau proposals whose energy has no bin number: NaN counts as
outside, below the histogram, and numbers past the integers' range as far
outside (the conversion saturates)."""
import numpy as np
import pytest

from cemc_amd.lattice import FCCSettings, random_occupation, seeded_ecis
from oracle.brute_force import brute_force_cf
from oracle.oracle import OracleModel, OracleUpdater

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("first", [True, False])
def test_nan_energies_are_outside(gpu, first):
    from cemc_amd.batch import ChainBatch
    from cemc_amd.model import CEModel
    s = FCCSettings(6, ["A", "B"], {2: 3, 3: 2})
    eci = seeded_ecis(s, 3, 0.02)
    eci[next(k for k in sorted(eci) if k.startswith("c2"))] = float("nan")
    batch = ChainBatch([CEModel(s, eci)], [dict(kind=0, temperature=900.0, seed=4, uid=0,
                                                occupation=random_occupation(s.n_sites, 2, 2))])
    batch.wl_set(0, 20, -1.0, 1.0, 1.0, current_bin=10, is_first=first)
    print("walker with NaN energies", first, flush=True)
    batch.wl_run(3, 100)
    got = batch.wl_get(0)
    assert (got["n_moves"], got["n_outside"], got["n_accept"]) == (300, 300, 0)
    assert not got["hist"].any() and not got["known"].any() and got["current_bin"] == 10


def test_energies_past_the_integers_range(gpu):
    from test_wang_landau import _centred, _gpu_vs_oracle
    s = FCCSettings(6, ["A", "B"], {2: 3, 3: 2})
    eci = seeded_ecis(s, 3, 1e6)
    occ = random_occupation(s.n_sites, 2, 2)
    names = s.cf_names()
    e0 = OracleUpdater(OracleModel(s, names), occ, brute_force_cf(s, occ, names), eci).get_energy()
    print("walker far outside", flush=True)
    got, _ = _gpu_vs_oracle(s, eci, occ, dict(_centred(e0, 1e-3, 20), f=1.0, cur_bin=10, is_first=False), 3, 100)
    assert got["n_outside"] > 250 and got["logdos"].sum() > 0  # counted once more from above


def test_range_narrower_than_the_smallest_bins(gpu):
    """A range of 1e-310: bins per eV overflow, and an energy at the lower end
    of the range still has bin 0 (all ECIs zero: every energy is 0)."""
    from test_wang_landau import _gpu_vs_oracle
    s = FCCSettings(6, ["A", "B"], {2: 3, 3: 2})
    eci = {k: 0.0 for k in seeded_ecis(s, 3, 1.0)}
    print("walker narrow range", flush=True)
    got, _ = _gpu_vs_oracle(s, eci, random_occupation(s.n_sites, 2, 2),
                            dict(n_bins=20, e_min=0.0, e_max=1e-310, f=1.0, cur_bin=10), 3, 100)
    assert got["n_accept"] > 0


def test_more_bins_than_the_lds_holds(gpu):
    """2^28 bins of 16 bytes are 2^32 bytes, which must not pass for none."""
    from cemc_amd.batch import ChainBatch
    from cemc_amd.model import CEModel
    s = FCCSettings(5, ["A", "B"], {2: 2})
    batch = ChainBatch([CEModel(s, seeded_ecis(s, 3, 0.02))],
                       [dict(kind=0, temperature=900.0, seed=4, uid=0, occupation=random_occupation(s.n_sites, 2, 2))])
    print("walker with 2^28 bins", flush=True)
    batch.wl_set(0, 1 << 28, -1.0, 1.0, 1.0)
    assert batch.wl_lanes_per_move(0) == 0
    with pytest.raises(ValueError, match="do not fit"):
        batch.wl_run(1, 10)
    batch.wl_set(0, 20, -1.0, 1.0, 1.0)
    batch.wl_run(1, 10)
    assert batch.wl_get(0)["n_moves"] == 10

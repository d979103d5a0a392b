"""Chains with constraints that depend on the proposal alone (fixed sites,
fixed species of canonical chains) and a bias on patch rounds of eight
(patch_kernel, kHook) against the oracle: fixed sites that need many
proposals, counts that run over a block's bias window, cells so small that
most rounds are cut, and a move without a valid proposal."""
import numpy as np
import pytest

from cemc_amd.lattice import FCCSettings, random_occupation, seeded_ecis
from oracle.brute_force import brute_force_cf
from oracle.oracle import OracleModel, OracleUpdater, run_hooked
from test_constraints import _bits, _gpu_vs_oracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kind,species,shells,size,share,fixed,slope", [
    (1, "AB", {2: 4, 3: 2}, 8, 0.1, 0, 40.0),
    (1, "AB", {2: 2}, 6, 0.7, 0, None),
    (1, "AB", {2: 2, 3: 1}, (3, 3, 4), 0.2, 0, 1.0),
    (1, "ABC", {2: 4, 3: 3, 4: 2}, 6, 0.3, 0, 5.0),
    (0, "AB", {2: 4, 3: 2}, 6, 0.5, 0, 1.0),
    (0, "ABC", {2: 4, 3: 3, 4: 2}, 6, 0.1, 2, None),
    (0, "ABCD", {2: 3, 3: 2}, 5, 0.3, 1, None),
])
def test_hooked_rounds_match_oracle(gpu, kind, species, shells, size, share, fixed, slope):
    S = len(species)
    s = FCCSettings(size, list(species), shells)
    rng = np.random.default_rng(6)
    allowed = np.where(rng.random(s.n_sites) < share, 0, 2 ** S - 1).astype(np.uint8)
    hooks = dict(allowed=allowed, fixed_species=fixed, max_attempts=400)
    if slope is not None:
        hooks.update(bias_species=0, bias_table=slope * (np.arange(s.n_sites + 1) / s.n_sites - 0.3) ** 2)
    occ = random_occupation(s.n_sites, S, 3)
    if slope == 40.0:
        occ[allowed != 0] = 1  # far from the bias' minimum: the count climbs
    print("hooked rounds", kind, species, size, share, fixed, slope, flush=True)
    batch, acc = _gpu_vs_oracle(s, seeded_ecis(s, 5, 0.01), occ, kind, 1500.0, 3000, hooks)
    assert batch.lanes_per_move(0) == 8
    assert acc > 50
    assert np.array_equal(batch.occupation(0)[allowed == 0], occ[allowed == 0])


@pytest.mark.parametrize("kind", [0, 1])
def test_hooked_rounds_stop_at_a_move_without_proposal(gpu, kind):
    from cemc_amd.batch import ChainBatch
    from cemc_amd.model import CEModel
    s = FCCSettings(6, ["A", "B"], {2: 3, 3: 2})
    eci = seeded_ecis(s, 5, 0.01)
    occ = random_occupation(s.n_sites, 2, 3)
    allowed = np.full(s.n_sites, 3, dtype=np.uint8)
    allowed[::8] = 0
    names = s.cf_names()
    hooks = dict(allowed=allowed, max_attempts=4 - kind)
    ora = OracleUpdater(OracleModel(s, names), occ, brute_force_cf(s, occ, names), eci)
    bits, _, acc, failed = run_hooked(ora, kind, 21, 4, 3000, 1500.0, **hooks)
    assert failed is not None and failed > 64
    batch = ChainBatch([CEModel(s, eci)], [dict(kind=kind, temperature=1500.0, occupation=occ, seed=21, uid=4)])
    batch.set_hooks(0, **hooks)
    print("hooked rounds stop", kind, "at move", failed, flush=True)
    with pytest.raises(RuntimeError, match="move %d" % failed):
        batch.run(3000)
    st = batch.stats()
    assert st["moves"][0] == failed and st["accepted"][0] == acc
    assert np.array_equal(batch.occupation(0), ora.get_occupation())
    assert abs(batch.energies()[0] - ora.get_energy()) / s.n_sites <= 1e-10

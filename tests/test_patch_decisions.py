"""Decisions of the patch kernel (cemc_amd/csrc/ce_patch_kernel.h) at the edge
of the acceptance threshold: u <= exp(-dE / kT) where dE differs from
-kT log u by less than the margin of the comparison on logarithms."""
import numpy as np
import pytest

from cemc_amd.lattice import KB_EV, FCCSettings, random_occupation, seeded_ecis
from oracle.oracle import philox4x64

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kind,species,chains,biased", [
    (0, "AB", 64, False),    # a row of lanes per move
    (1, "AB", 64, False),
    (0, "AB", 1100, False),  # a quad per move
    (1, "ABC", 64, False),
    (0, "ABC", 64, False),
    (1, "AB", 64, True),     # one after the other, with the bias
])
def test_margin_decisions_use_the_chains_temperature(gpu, kind, species, chains, biased):
    """One move per chain.  At a temperature where dE is (1 + 1e-12) times the
    threshold, relative to kT + dE, u exceeds the probability; on the other side
    it does not.  The margin is 2e-12; dE from the energies before and after
    is good to 1e-13 of itself."""
    from cemc_amd.batch import ChainBatch
    from cemc_amd.model import CEModel
    s = FCCSettings(6, list(species), {2: 4, 3: 2})
    model = CEModel(s, seeded_ecis(s, 3, 0.05))
    occ = random_occupation(s.n_sites, len(species), 2)
    bias = 8.0 * ((np.arange(s.n_sites + 1) - 60.0) / s.n_sites) ** 2

    def after_one_move(temps):
        batch = ChainBatch([model] * chains, [dict(kind=kind, temperature=float(t), occupation=occ, seed=11, uid=c)
                                              for c, t in enumerate(temps)])
        batch.set_patches(True)
        if biased:
            for c in range(chains):
                batch.set_hooks(c, bias_species=0, bias_table=bias)
        assert batch.lanes_per_move(0) == (8 if biased else (4 if chains > 512 else 16))
        e0 = batch.energies()
        batch.run(1)
        return batch.stats()["accepted"], batch.energies() - e0

    print("margin", kind, species, chains, biased, flush=True)
    acc, de = after_one_move(np.full(chains, 1e9))  # kT = 86000 eV: every move is made
    assert acc.all()
    u = np.array([(philox4x64((0, 0, 0, 0), (11, c))[3] >> 11) * 2.0 ** -53 for c in range(chains)])
    x = -np.log(u)
    use = (de > 0.02) & (u > 0.02) & (u < 0.7)
    assert use.sum() >= 6
    for side in (1.0, -1.0):
        temps = np.where(use, de / (KB_EV * (x + side * 1e-12 * (1.0 + x))), 1000.0)
        acc, _ = after_one_move(temps)
        assert np.array_equal(acc[use] == 0, np.full(use.sum(), side > 0))

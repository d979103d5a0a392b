"""Lattices read back through the read-back kernel (up to 8 KB) and past its
limit: sizes that are no multiple of a word, a second chain at whatever offset
the first one leaves it, the last size below the limit and the first above."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("size", [(3, 3, 5), (5, 5, 7), (16, 16, 16), (32, 16, 16), (21, 21, 19)])
def test_lattices_read_back(gpu, size):
    from cemc_amd.batch import ChainBatch
    from cemc_amd.lattice import FCCSettings, random_occupation, seeded_ecis
    from cemc_amd.model import CEModel
    s = FCCSettings(size, ["A", "B", "C"], {2: 1})
    occ = [random_occupation(s.n_sites, 3, 5 + c) for c in range(2)]
    print("read back", s.n_sites, "sites", flush=True)
    batch = ChainBatch([CEModel(s, seeded_ecis(s, 1, 0.01))] * 2,
                       [dict(kind=1, temperature=500.0, occupation=o, seed=1, uid=c,
                             chem_pot={"c1_0": 0.0, "c1_1": 0.0}) for c, o in enumerate(occ)])
    for c in (1, 0):
        assert np.array_equal(batch.occupation(c), occ[c])
    batch.run(200)
    for c in range(2):
        changed = np.count_nonzero(batch.occupation(c) != occ[c])
        assert 0 < changed <= batch.stats()["accepted"][c]

"""Lattices from translation tables on the sweep kernel: the table in LDS or,
where it does not fit, in memory; at most one record per lane, two, or more
(lds_move_de and the batches of lds_flip_de); both move kinds, against the
oracle move for move."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kind", [0, 1])
@pytest.mark.parametrize("size,species,shells,records", [
    ((4, 4, 4), "ABC", {2: 1.45, 3: 1.05, 4: 1.05}, (1, 64)),
    ((4, 4, 4), "ABC", {2: 1.75, 3: 1.45}, (65, 128)),
    ((4, 4, 4), "AB", {2: 1.75, 3: 1.45, 4: 1.45}, (129, 10000)),
    ((14, 14, 12), "AB", {2: 1.45, 3: 1.05}, (1, 64)),
])
def test_table_lattice_chains_match_oracle(gpu, kind, size, species, shells, records):
    from cemc_amd.batch import ChainBatch
    from cemc_amd.crystal import HCPSettings
    from cemc_amd.lattice import random_occupation, seeded_ecis
    from cemc_amd.model import CEModel
    from oracle.brute_force import brute_force_cf
    from oracle.oracle import OracleModel, OracleUpdater
    s = HCPSettings(size, list(species), shells)
    per_site = max(sum(len(c["indices"]) for c in g.values() if c["size"] > 1) for g in s.cluster_info)
    assert records[0] <= per_site <= records[1]
    eci = seeded_ecis(s, 5, 0.01)
    occ = random_occupation(s.n_sites, len(species), 3)
    n = 3000
    print("table lattice", kind, size, species, per_site, "records", flush=True)
    batch = ChainBatch([CEModel(s, eci)], [dict(kind=kind, temperature=900.0, occupation=occ, seed=3, uid=1)])
    log = batch.run_logged(n)
    names = s.cf_names()
    ora = OracleUpdater(OracleModel(s, names), occ, brute_force_cf(s, occ, names), eci)
    bits, _, acc = ora.run(kind, 3, 1, n, 900.0)

    def unpack(b):
        return np.unpackbits(np.asarray(b, dtype=np.uint8), bitorder="little")[:n]

    assert acc > 100 and np.array_equal(unpack(log[0]), unpack(bits))
    assert np.array_equal(batch.occupation(0), ora.get_occupation())
    assert abs(batch.energies()[0] - ora.get_energy()) / s.n_sites <= 1e-10

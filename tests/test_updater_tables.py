"""Changes of the correlation functions through the updater's product tables:
tables in LDS, tables read from memory, and models past the size limit of the
tables (one product per decoration), each against the oracle, in calls of one
change and of two, with the resident kernel and with a launch per call."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("species,shells,every,lo,hi", [
    ("ABC", {2: 3, 3: 2, 4: 1}, 1, 1, 16384),
    ("ABCD", {2: 2, 3: 2, 4: 2}, 1, 16384, 1 << 20),
    ("ABCDEFGH", {2: 1, 3: 1, 4: 1}, 2, 1 << 20, 1 << 30),
])
def test_updater_tables_match_oracle(gpu, species, shells, every, lo, hi):
    from cemc_amd.lattice import FCCSettings, SimpleAtoms, random_occupation
    from cemc_amd.updater import PyCEUpdater
    from oracle.brute_force import brute_force_cf
    from oracle.oracle import OracleModel, OracleUpdater
    S = len(species)
    s = FCCSettings(4, list(species), shells)
    names = s.cf_names()
    names = sorted({n for n in names if not n.startswith("c4")} | set(names[::every]))
    doubles = sum(int(n[1]) * (S - 1) * S ** (int(n[1]) - 1) for n in names if n[1] in "234")
    assert lo <= doubles < hi
    rng = np.random.default_rng(8)
    eci = {n: float(rng.uniform(-0.01, 0.01)) for n in names}
    occ = random_occupation(s.n_sites, S, 21)
    cf0 = brute_force_cf(s, occ, names)
    print("updater tables", species, len(names), "functions", doubles, "doubles", flush=True)
    runs = []
    for resident in (True, False):
        upd = PyCEUpdater(SimpleAtoms([s.species[v] for v in occ]), s, cf0, eci)
        upd.set_resident(resident)
        ora = OracleUpdater(OracleModel(s, names), occ, cf0, eci)
        step_rng = np.random.default_rng(4)
        cur, got = [int(v) for v in occ], []
        for step in range(30):
            i, j = (int(v) for v in step_rng.choice(s.n_sites, 2, replace=False))
            to = (cur[i] + 1 + step) % S
            to = to if to != cur[i] else (to + 1) % S
            chs = [(i, s.species[cur[i]], s.species[to])]
            if step % 3:
                chs.append((j, s.species[cur[j]], s.species[(cur[j] + 1) % S]))
            got.append(upd.calculate(chs))
            # 4800 products of at most 1e-2 x 64 sites: 1e-12 per site as elsewhere
            assert abs(got[-1] - ora.calculate(chs)) / s.n_sites <= 1e-12
            if step % 4 == 1:
                upd.undo_changes()
                ora.undo_changes()
            else:
                upd.clear_history()
                ora.clear_history()
            cur = [int(v) for v in ora.get_occupation()]
            assert np.max(np.abs(upd.get_cf_array() - ora.get_cf_array())) <= 1e-12
        upd.close()
        runs.append(got)
    assert runs[0] == runs[1]

"""Models at the edge of what the patch kernel takes, against the oracle."""
import copy

import numpy as np
import pytest

from cemc_amd.lattice import FCCSettings, random_occupation, seeded_ecis
from oracle.brute_force import brute_force_cf
from oracle.oracle import OracleModel, OracleUpdater

pytestmark = pytest.mark.gpu


def _chains_vs_oracle(s, eci, kind, temperature, n_moves, chains=1, always=True):
    from cemc_amd.batch import ChainBatch
    from cemc_amd.model import CEModel
    S = len(s.unique_elements)
    occ = random_occupation(s.n_sites, S, 3)
    batch = ChainBatch([CEModel(s, eci)] * chains,
                       [dict(kind=kind, temperature=temperature, occupation=occ, seed=3, uid=c) for c in range(chains)])
    batch.set_patches(always)
    log = batch.run_logged(n_moves)
    names = s.cf_names()
    for c in {0, chains - 1}:
        ora = OracleUpdater(OracleModel(s, names), occ, brute_force_cf(s, occ, names), eci)
        bits, _, acc = ora.run(kind, 3, c, n_moves, temperature)
        assert 0 < acc < n_moves
        assert np.array_equal(np.unpackbits(log[c], bitorder="little")[:n_moves],
                              np.unpackbits(bits, bitorder="little")[:n_moves])
        assert np.array_equal(batch.occupation(c), ora.get_occupation())
    return batch


@pytest.mark.parametrize("kind", [0, 1])
def test_one_sided_sub_clusters(gpu, kind):
    """Pairs listed for one of their two sites only: a change at a site reaches
    flips on one side of it, so a move past a blocked one may write what the
    blocked one reads."""
    s = copy.copy(FCCSettings((5, 5, 6), ["A", "B"], {2: 2}))
    info = s.cluster_info[0]
    dims = np.array(s.dims)
    for name, cl in info.items():
        if cl["size"] != 2:
            continue
        # keep the member whose wrapped offset comes first of +o and -o
        keep = [k for k, sub in enumerate(cl["indices"])
                if tuple(s.cells[sub[0]]) < tuple((-np.array(s.cells[sub[0]])) % dims)]
        assert 2 * len(keep) == len(cl["indices"])
        cl["indices"] = [cl["indices"][k] for k in keep]
        cl["order"] = [cl["order"][k] for k in keep]
    print("one-sided pairs", kind, flush=True)
    batch = _chains_vs_oracle(s, seeded_ecis(s, 5, 0.02), kind, 1200.0, 6000)
    assert batch.lanes_per_move(0) == 0


@pytest.mark.parametrize("kind", [0, 1])
@pytest.mark.parametrize("size,lanes", [((127, 5, 5), 16), ((128, 5, 5), 0), ((5, 5, 127), 16), ((5, 128, 5), 0)])
def test_longest_axes(gpu, kind, size, lanes):
    """Cell differences of the pair test take a byte per axis, up to 253 at 127
    cells; longer lattices run on the sweep kernel."""
    s = FCCSettings(size, ["A", "B"], {2: 4, 3: 2})
    print("longest axes", size, kind, flush=True)
    batch = _chains_vs_oracle(s, seeded_ecis(s, 5, 0.02), kind, 1200.0, 6000)
    assert batch.lanes_per_move(0) == lanes


@pytest.mark.parametrize("kind", [0, 1])
def test_more_patches_than_the_kernel_takes(gpu, kind):
    """1001 patches (448 at most): the sweep kernel."""
    s = FCCSettings(5, ["A", "B", "C", "D"], {2: 4, 3: 4, 4: 4})
    print("many patches", kind, flush=True)
    batch = _chains_vs_oracle(s, seeded_ecis(s, 5, 0.005), kind, 1200.0, 600)
    assert batch.lanes_per_move(0) == 0


@pytest.mark.parametrize("size,kind,temperature,chains,lanes", [
    (5, 0, 2500.0, 1, 0),     # every swap reaches most of the cell, most are made
    (5, 0, 250.0, 1, 16),     # few are made
    (5, 1, 2500.0, 1, 16),    # a flip reaches 0.44 of the cell
    (5, 1, 2500.0, 600, 0),
    (8, 0, 1000.0, 4, 16),
    (6, 0, 700.0, 1100, 0),   # more chains than SIMDs: conflicts cost more
    (10, 0, 700.0, 1100, 4),
])
def test_chains_whose_moves_mostly_conflict(gpu, size, kind, temperature, chains, lanes):
    """Small cells at high acceptance run one move at a time."""
    s = FCCSettings(size, ["A", "B"], {2: 4, 3: 2})
    print("conflicting chains", size, kind, temperature, chains, flush=True)
    batch = _chains_vs_oracle(s, seeded_ecis(s, 3, 0.02), kind, temperature, 500, chains, always=False)
    assert batch.lanes_per_move(0) == lanes


def test_a_temperature_that_changes_the_kernel(gpu):
    """Annealing a small cell: one move at a time while it is hot, then the
    patch kernel, move for move the oracle's."""
    from cemc_amd.batch import ChainBatch
    from cemc_amd.model import CEModel
    s = FCCSettings(5, ["A", "B"], {2: 4, 3: 2})
    eci = seeded_ecis(s, 3, 0.02)
    occ = random_occupation(s.n_sites, 2, 3)
    names = s.cf_names()
    ora = OracleUpdater(OracleModel(s, names), occ, brute_force_cf(s, occ, names), eci)
    batch = ChainBatch([CEModel(s, eci)], [dict(kind=0, temperature=2500.0, occupation=occ, seed=3, uid=0)])
    done = 0
    print("annealing", flush=True)
    for temperature, lanes in ((2500.0, 0), (300.0, 16), (290.0, 16), (2000.0, 0)):
        batch.set_temperature(0, temperature)
        batch.run(777)
        assert batch.lanes_per_move(0) == lanes
        ora.run(0, 3, 0, 777, temperature, move_begin=done)
        done += 777
        assert np.array_equal(batch.occupation(0), ora.get_occupation())
        assert abs(batch.energies()[0] - ora.get_energy()) <= 1e-10 * s.n_sites


def test_pools_whose_chains_conflict(gpu):
    """A pool of small hot cells runs one move at a time, a mixed one does not
    split its launches."""
    from cemc_amd.batch import ChainPool
    from cemc_amd.model import CEModel
    s = FCCSettings(5, ["A", "B"], {2: 4, 3: 2})
    model = CEModel(s, seeded_ecis(s, 3, 0.02))
    occ = random_occupation(s.n_sites, 2, 3)
    n = 20
    pool = ChainPool(n, 1, n * 128, n * 128)
    for c in range(n):
        assert pool.add(model, dict(kind=0, temperature=2500.0, occupation=occ, seed=3, uid=c)) == c
    print("pools", flush=True)
    for cold, lanes in ((0, 0), (2, 0), (3, 16)):
        for c in range(cold):
            pool.set_temperature(c, 250.0)
        pool.run(np.full(n, 100, dtype=np.int64))
        assert pool.lanes_per_move(n - 1) == lanes


def test_pools_with_empty_slots(gpu):
    """Launches of a pool that never had a chain, and of one whose chains left."""
    from cemc_amd.batch import ChainPool
    from cemc_amd.model import CEModel
    s = FCCSettings(5, ["A", "B"], {2: 4, 3: 2})
    pool = ChainPool(4, 1, 4 * 128, 4 * 128)
    print("empty pool", flush=True)
    pool.run(np.zeros(4, dtype=np.int64))
    model = CEModel(s, seeded_ecis(s, 3, 0.02))
    c = pool.add(model, dict(kind=0, temperature=900.0, occupation=random_occupation(s.n_sites, 2, 3), seed=3, uid=0))
    pool.run(np.where(np.arange(4) == c, 100, 0))
    assert pool.stats()["moves"][c] == 100
    pool.remove(c)
    pool.run(np.zeros(4, dtype=np.int64))

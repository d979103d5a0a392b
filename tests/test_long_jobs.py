"""A pool's longest job on a crowded device: it gets four waves, also on the
patch kernel (but not for flips with at most 16 patches, where one wave is
faster), and ends where it ends alone."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("species,shells,kind,waves", [
    ("AB", {2: 4, 3: 2}, 0, 4),
    ("AB", {2: 4, 3: 2}, 1, 1),
    ("ABC", {2: 4, 3: 3, 4: 2}, 1, 4),
    ("ABCD", {2: 3, 3: 3, 4: 3}, 0, 4),
])
def test_long_job_in_a_crowd(gpu, species, shells, kind, waves):
    from cemc_amd.batch import ChainBatch, ChainPool
    from cemc_amd.lattice import FCCSettings, random_occupation, seeded_ecis
    from cemc_amd.model import CEModel
    s = FCCSettings(6, list(species), shells)
    model = CEModel(s, seeded_ecis(s, 3, 0.02))
    occ = random_occupation(s.n_sites, len(species), 1)
    n = 1100
    pool = ChainPool(n, 1, n * 512, n * 512)
    pool.set_patches(True)
    print("long job", species, kind, flush=True)
    moves = np.full(n, 64, dtype=np.int64)
    for c in range(n):
        assert pool.add(model, dict(kind=kind, temperature=900.0, occupation=occ, seed=5, uid=c)) == c
    moves[700] = 1 << 21
    pool.run_sliced(moves, 1.0)
    assert pool.launch_shape(700)[0] == waves
    assert pool.lanes_per_move(700) == (4 if waves == 1 else (64 if len(species) == 4 else 16))
    assert pool.launch_shape(0)[0] == (1 if len(species) < 4 else 2)
    done = pool.stats()["moves"]
    assert 64 < done[700] < moves[700] and done[0] == 64
    alone = ChainBatch([model], [dict(kind=kind, temperature=900.0, occupation=occ, seed=5, uid=700)])
    alone.run(int(done[700]))
    assert np.array_equal(alone.occupation(0), pool.occupation(700))
    assert alone.stats()["accepted"][0] == pool.stats()["accepted"][700]

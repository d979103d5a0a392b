"""Runs on the patch kernel cut into launches end bitwise where one run ends:
lattices, energies, moves and accepted moves; sample sums to rounding, since
each launch adds its partial sums to the chain's.  Cut at arbitrary moves,
and by the time limit of slices (chains of one and of several waves)."""
import numpy as np
import pytest

from cemc_amd.lattice import FCCSettings, random_occupation, seeded_ecis

pytestmark = pytest.mark.gpu


def _batch(species, shells, size, kind, n, hooked=False):
    from cemc_amd.batch import ChainBatch
    from cemc_amd.model import CEModel
    s = FCCSettings(size, list(species), shells)
    model = CEModel(s, seeded_ecis(s, 5, 0.02))
    mu = {"c1_0": 0.01} if kind else {}
    occ = random_occupation(s.n_sites, len(species), 4)
    make = lambda: ChainBatch([model] * n, [dict(kind=kind, temperature=400.0 + 2000.0 * c / n, occupation=occ,  # noqa: E731
                                                 seed=6, uid=c, chem_pot=mu) for c in range(n)])
    batches = make(), make()
    for b in batches:
        b.set_patches(True)
    if hooked:
        allowed = np.where(np.arange(s.n_sites) % 10 == 0, 0, 2 ** len(species) - 1).astype(np.uint8)
        for b in batches:
            for c in range(n):
                b.set_hooks(c, allowed=allowed, bias_species=0, bias_table=np.arange(s.n_sites + 1) ** 2 * 1e-4)
    return batches


def _assert_same(a, b, chains):
    sa, sb = a.stats(), b.stats()
    assert np.array_equal(sa["moves"], sb["moves"]) and np.array_equal(sa["accepted"], sb["accepted"])
    assert np.array_equal(a.energies(), b.energies())
    for c in chains:
        assert np.array_equal(a.occupation(c), b.occupation(c))
    for key in ("sum_e", "sum_e2"):
        np.testing.assert_allclose(sa[key], sb[key], rtol=1e-12, atol=1e-9)


@pytest.mark.parametrize("species,shells,size,kind,n,hooked", [
    ("AB", {2: 4, 3: 2}, 8, 0, 3, False),
    ("AB", {2: 4, 3: 2}, 6, 1, 1100, False),
    ("ABC", {2: 4, 3: 3, 4: 2}, 6, 0, 1100, False),
    ("ABC", {2: 4, 3: 3, 4: 2}, 6, 1, 3, False),
    ("ABCD", {2: 3, 3: 3, 4: 3}, 6, 0, 2, False),
    ("AB", {2: 4, 3: 2}, 8, 1, 5, True),
])
def test_energies_do_not_depend_on_where_launches_end(gpu, species, shells, size, kind, n, hooked):
    whole, parts = _batch(species, shells, size, kind, n, hooked)
    print("split", species, kind, n, whole.launch_shape(0), flush=True)
    assert whole.lanes_per_move(0) > 0
    cuts = [1, 7, 0, 64, 100, 28, 333]
    whole.run(sum(cuts))
    for m in cuts:
        parts.run(m)
    _assert_same(whole, parts, {0, n // 2, n - 1})


@pytest.mark.parametrize("species,shells,kind,n,waves", [
    ("AB", {2: 4, 3: 2}, 0, 1, 4),
    ("AB", {2: 4, 3: 2}, 1, 1100, 1),
    ("ABC", {2: 4, 3: 3, 4: 2}, 0, 300, 2),
    ("ABCD", {2: 3, 3: 3, 4: 3}, 1, 1, 8),
])
def test_time_slices_continue_each_chains_stream(gpu, species, shells, kind, n, waves):
    whole, slices = _batch(species, shells, 8, kind, n)
    assert whole.launch_shape(0)[0] == waves and whole.lanes_per_move(0) > 0
    moves = 12000
    print("slices", species, kind, n, flush=True)
    whole.run(moves)
    launches = 0
    while True:
        left = moves - slices.stats()["moves"]
        if left.max() == 0:
            break
        assert left.min() >= 0 and launches < 5000
        slices.run_sliced(left, 0.1)
        launches += 1
    assert launches > 2
    _assert_same(whole, slices, {0, n // 2, n - 1})


def test_a_state_changed_between_launches(gpu):
    """A launch that ends inside a block, then a bias that shifts the energy, a
    run on the sweep kernel or other chains in the slot: the next launch goes
    on from the energy as it is."""
    from cemc_amd.batch import ChainBatch
    from cemc_amd.model import CEModel
    s = FCCSettings(6, ["A", "B"], {2: 4, 3: 2})
    model = CEModel(s, seeded_ecis(s, 5, 0.02))
    occ = random_occupation(s.n_sites, 2, 4)
    print("state changed between launches", flush=True)
    b = ChainBatch([model], [dict(kind=1, temperature=900.0, occupation=occ, seed=6, uid=0, first_move=37)])
    table = np.arange(s.n_sites + 1) * 0.01
    b.set_patches(True)
    for step in range(4):
        b.run(41)
        if step == 1:
            b.set_hooks(0, bias_species=0, bias_table=table)
        if step == 2:
            b.clear_hooks(0)
            b.set_waves(1)  # the sweep kernel
            b.run(13)
            b.set_waves(0)
        e, exact = b.energies()[0], b.cf(0)[1]
        if step == 1:
            exact += table[b.hooks_state(0)[1]]
        assert abs(e - exact) <= 1e-12 * s.n_sites

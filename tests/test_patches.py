"""The regrouping of a site's sub-clusters into patches
(cemc_amd/csrc/ce_patches.h) on the CPU: for random tables and random
neighbourhoods the patch entries sum to the sub-clusters' entries, whatever
the lattice, the cluster set, the species count and the decoration symmetry.
On the GPU, the patch kernel against the oracle at its edges."""
import itertools
import os
import subprocess

import numpy as np
import pytest

from cemc_amd.crystal import HCPSettings
from cemc_amd.lattice import CubicSettings, FCCSettings, random_occupation, seeded_ecis
from oracle.brute_force import brute_force_cf
from oracle.oracle import OracleModel, OracleUpdater

HERE = os.path.dirname(os.path.abspath(__file__))


@pytest.fixture(scope="module")
def search(tmp_path_factory):
    exe = str(tmp_path_factory.mktemp("patch") / "patch_check")
    subprocess.run(["g++", "-O2", "-std=c++17", os.path.join(HERE, "patch_check.cpp"), "-o", exe], check=True)
    return exe


def _records(settings, group):
    """(member columns, block name, equivalent member orders) per sub-cluster,
    the reference site brought to the lowest position it may take."""
    out = []
    for name, cl in settings.cluster_info[group].items():
        n = int(cl["size"])
        if n < 2:
            continue
        same = [p for p in itertools.permutations(range(n))
                if all(i == p[i] or any(i in g and p[i] in g for g in cl["equiv_sites"]) for i in range(n))]
        for sub, order in zip(cl["indices"], cl["order"]):
            at = [None if k == 0 else int(sub[k - 1]) for k in order]
            perm = min(same, key=lambda p: p[at.index(None)])
            now = [None] * n
            for pos in range(n):
                now[perm[pos]] = at[pos]
            ref = now.index(None)
            place = [pos for pos in range(n) if pos != ref]
            orders = [[place.index(p[pos]) for pos in place] for p in same if p[ref] == ref]
            out.append(([c for c in now if c is not None], (name, ref), orders))
    return out


@pytest.mark.parametrize("make,species,q", [
    (lambda sp: FCCSettings(10, sp, {2: 4, 3: 2}), 2, 6),
    (lambda sp: FCCSettings(10, sp, {2: 4}), 2, 6),
    (lambda sp: FCCSettings(8, sp, {2: 4, 3: 3, 4: 2}), 3, 5),
    (lambda sp: FCCSettings(8, sp, {2: 3, 3: 2, 4: 1}, symmetrize_decorations=False), 3, 5),
    (lambda sp: FCCSettings(8, sp, {2: 3, 3: 3, 4: 3}), 4, 4),
    (lambda sp: CubicSettings(7, sp, {2: 3, 3: 2, 4: 1}, lattice="bcc"), 3, 5),
    (lambda sp: CubicSettings(7, sp, {2: 3, 3: 2, 4: 1}, lattice="sc"), 4, 4),
    (lambda sp: HCPSettings((4, 4, 3), sp, {2: 1.45, 3: 1.05, 4: 1.05}), 3, 5),
])
def test_patch_entries_sum_to_the_subclusters_entries(search, make, species, q):
    st = make(list("ABCD"[:species]))
    recs = _records(st, 0)
    rng = np.random.default_rng(5)
    cols = sorted({c for mem, _, _ in recs for c in mem})
    bits = 1 if species == 2 else 2
    width = (species - 1) << (3 * bits)
    blocks = {}
    tables = []
    for mem, name, orders in recs:
        if name in blocks:
            continue
        blocks[name] = len(tables) * width
        n = len(mem)
        # random entries per species of the members, alike under the
        # equivalent orders (slot m shows member o[m])
        g = rng.normal(size=(species - 1,) + (species,) * n)
        g = sum(np.transpose(g, [0] + [1 + int(np.argsort(o)[m]) for m in range(n)]) for o in orders)
        flat = np.zeros((species - 1, 1 << (3 * bits)))
        for d in range(species - 1):
            for sp in itertools.product(range(species), repeat=n):
                flat[d, sum(s << (bits * m) for m, s in enumerate(sp))] = g[(d,) + sp]
        tables.append(flat.ravel())
    rec_tab = np.concatenate(tables)
    lines = ["%d %d %d %d %d %d" % (len(cols), len(recs), q, species, bits, rec_tab.size)]
    for mem, name, orders in recs:
        ids = [cols.index(c) for c in mem] + [-1] * (3 - len(mem))
        orders = [list(o) + list(range(len(o), 3)) for o in orders]
        lines.append(" ".join(str(v) for v in [len(mem)] + ids + [blocks[name], len(orders)] + sum(orders, [])))
    lines.append(" ".join("%.17g" % v for v in rec_tab))
    got = subprocess.run([search], input="\n".join(lines), capture_output=True, text=True, check=True).stdout.split("\n")
    n_patch, n_tab = (int(v) for v in got[0].split())
    patches = np.array([[int(v) for v in ln.split()] for ln in got[1:1 + n_patch]])
    tabs = [np.array([float(v) for v in ln.split()]).reshape(species ** q, species - 1)
            for ln in got[1 + n_patch:1 + n_patch + n_tab]]
    assert 0 < n_patch < len(recs)
    assert patches[:, q].max() == n_tab - 1
    for _ in range(50):
        occ = rng.integers(species, size=len(cols))
        want = np.zeros(species - 1)
        for mem, name, _ in recs:
            code = sum(int(occ[cols.index(c)]) << (bits * m) for m, c in enumerate(mem))
            want += rec_tab[[blocks[name] + (d << (3 * bits)) + code for d in range(species - 1)]]
        have = np.zeros(species - 1)
        for p in patches:
            # a place that the patch does not use may show any species
            sp = [occ[s] if s >= 0 else rng.integers(species) for s in p[:q]]
            have += tabs[p[q]][sum(int(s) * species ** i for i, s in enumerate(sp))]
        # both are sums of at most 1746 entries of order one
        np.testing.assert_allclose(have, want, rtol=0, atol=1e-11)


@pytest.mark.gpu
@pytest.mark.parametrize("kind", [0, 1])
@pytest.mark.parametrize("species,shells,size,symm,chains,lanes,waves,per_lane", [
    (2, {2: 4, 3: 2}, 10, True, 1, 16, 4, 1),             # 12 patches
    (2, {2: 4, 3: 2}, (5, 7, 6), True, 700, 4, 1, 3),     # smallest box of the halo, one wave each
    (2, {2: 4, 3: 3, 4: 2}, 5, True, 300, 16, 2, 4),      # 47 patches, two waves
    (3, {2: 3, 3: 2}, (6, 5, 9), False, 3, 16, 4, 1),     # no shared tables
    (3, {2: 4, 3: 3, 4: 2}, 9, True, 2, 16, 4, 4),        # 59 patches, four waves
    (3, {2: 4, 3: 3, 4: 2}, 5, True, 600, 4, 1, 15),
    (4, {2: 3, 3: 2, 4: 1}, (5, 6, 5), True, 2, 16, 4, 2),
    (4, {2: 3, 3: 3, 4: 3}, 5, True, 1, 64, 8, 7),        # 426 patches, eight waves
    (4, {2: 3, 3: 3, 4: 3}, 6, True, 300, 64, 2, 7),      # and two
    (4, {2: 3, 3: 2}, (5, 6, 5), True, 600, 4, 1, 6),     # 24 patches, a quad each
    (4, {2: 3, 3: 2, 4: 1}, 5, True, 600, 4, 1, 9),       # 32
    (2, {2: 3, 3: 3, 4: 3}, 5, True, 1, 64, 8, 4),        # 164 patches, a wave per move: eight waves
    (2, {2: 3, 3: 3, 4: 3}, 5, True, 200, 64, 4, 4),      # and four
    (3, {2: 4, 3: 4}, 5, True, 1, 64, 8, 2),              # 96 patches
    (3, {2: 3, 3: 3, 4: 3}, 5, True, 300, 64, 2, 4),      # 220
    (4, {2: 3, 3: 3}, 5, True, 200, 64, 4, 2),            # 84
])
def test_patch_kernel_matches_oracle(gpu, kind, species, shells, size, symm, chains, lanes, waves, per_lane):
    """Flips, and swaps whose sites interact (small cells), in launches that
    end inside a round and a block: accept bits and lattices equal the
    oracle's, energies and sample sums to rounding."""
    from cemc_amd.batch import ChainBatch
    from cemc_amd.model import CEModel
    st = FCCSettings(size, list("ABCD"[:species]), shells, symmetrize_decorations=symm)
    eci = seeded_ecis(st, 31, 0.02)
    names = st.cf_names()
    occ = random_occupation(st.n_sites, species, 6)
    temps = np.geomspace(400.0, 2500.0, chains) if chains > 1 else [900.0]
    mu = {"c1_%d" % d: 0.02 * (d + 1) for d in range(species - 1)} if kind else {}
    batch = ChainBatch([CEModel(st, eci)] * chains,
                       [dict(kind=kind, temperature=float(t), occupation=occ, seed=8, uid=c, chem_pot=mu)
                        for c, t in enumerate(temps)])
    batch.set_patches(True)
    print("patches", species, shells, size, "kind", kind, "chains", chains, batch.launch_shape(0), flush=True)
    assert batch.lanes_per_move(0) == lanes
    assert batch.launch_shape(0)[:2] == (waves, per_lane)
    parts = [1, 7, 64, 65, 330]
    logs = [batch.run_logged(n) for n in parts]
    total = sum(parts)
    stats, energies = batch.stats(), batch.energies()
    cf0 = brute_force_cf(st, occ, names)
    for c in sorted({0, chains // 2, chains - 1}):
        ora = OracleUpdater(OracleModel(st, names), occ, cf0, {k: v - mu.get(k, 0.0) for k, v in eci.items()})
        bits, trace, singlets, acc = [], [], [], 0
        for t in range(total):
            bit, e, a = ora.run(kind, 8, c, 1, float(temps[c]), move_begin=t, trace_every=1)
            bits.append(bit[0] & 1)
            trace.append(e[0])
            acc += a
            if kind:
                cf = ora.get_cf()
                singlets.append([cf["c1_%d" % d] for d in range(species - 1)])
        got = np.concatenate([np.unpackbits(lg[c], bitorder="little")[:n] for lg, n in zip(logs, parts)])
        assert np.array_equal(got, bits)
        assert np.array_equal(batch.occupation(c), ora.get_occupation())
        assert stats["accepted"][c] == acc
        # 1e-12 eV a site: 467 additions of changes below 1 eV round to 1e-13 eV
        assert abs(energies[c] - ora.get_energy()) <= 1e-12 * st.n_sites
        assert abs(stats["sum_e"][c] - np.sum(trace)) <= 1e-12 * st.n_sites * total
        th = batch.thermo(c)
        assert abs(th["mean_energy"] - np.mean(trace)) <= 1e-12 * st.n_sites
        if kind:
            np.testing.assert_allclose(th["singlet"], np.mean(singlets, axis=0), rtol=0, atol=1e-12)
            np.testing.assert_allclose(th["var_singlet"], np.var(singlets, axis=0), rtol=0, atol=1e-12)
            cov = np.mean(np.array(singlets) * np.array(trace)[:, None], axis=0) - th["singlet"] * np.mean(trace)
            np.testing.assert_allclose(th["cov_singlet_energy"], cov, rtol=0, atol=1e-11 * st.n_sites)


@pytest.mark.gpu
@pytest.mark.parametrize("species,shells,size,half,bins", [
    (2, {2: 4, 3: 2}, (5, 6, 7), 0.7, 33),          # two patches a lane, narrow range
    (2, {2: 4, 3: 3, 4: 2}, 5, 3.0, 100),           # eight
    (3, {2: 4, 3: 3, 4: 2}, 6, 0.4, 7),             # few bins, many proposals outside
    (4, {2: 3, 3: 2, 4: 1}, (6, 5, 5), 2.0, 1000),  # four, most bins unvisited
])
def test_patch_walkers_match_oracle(gpu, species, shells, size, half, bins):
    """Wang-Landau swaps on the patch kernel, checks that end inside a block:
    histogram, ln g (bit for bit), f and lattice equal the oracle's."""
    from test_wang_landau import _centred, _gpu_vs_oracle
    s = FCCSettings(size, list("ABCD"[:species]), shells)
    eci = seeded_ecis(s, 12, 0.02)
    occ = random_occupation(s.n_sites, species, 4)
    names = s.cf_names()
    e0 = OracleUpdater(OracleModel(s, names), occ, brute_force_cf(s, occ, names), eci).get_energy()
    print("patch walker", species, shells, size, flush=True)
    got, batch = _gpu_vs_oracle(s, eci, occ, dict(_centred(e0, half, bins), f=1.0, f_min=1e-3, flatness=0.3,
                                                  cur_bin=bins // 2), 9, 333)
    assert got["n_accept"] > 0
    assert batch.wl_lanes_per_move(0) == 8 and batch.wl_lanes_per_move(0, shared=True) == 0

"""What is measured of this framework's speed.

Each case is work that a user has the framework do, through its public entry
points: single changes through the updater, Metropolis chains (one, many of
one size, many of mixed sizes and ensembles, constrained ones, on closed-form
and on general lattices), replica exchange, Wang-Landau walkers and
correlation functions from scratch.  Sizes and interactions are those of the
repository's benchmark, job stream and tests.

A sampler's pass ends as a user's does: the energies, the accept counts and
the sample sums of every chain and every chain's final lattice are read back.
"""
import itertools
import math

import numpy as np

KB = 8.617330337217213e-05  # eV/K

# Interactions: largest neighbour shell per cluster size on cubic lattices,
# largest diameter per size on HCP (units of a), and the ECI spread in eV.
INTERACTIONS = {
    "pairs": ({2: 2}, 0.02),
    "pairs_triplets": ({2: 4, 3: 2}, 0.02),
    "four_body": ({2: 4, 3: 3, 4: 2}, 0.01),
    "third_shell": ({2: 3, 3: 3, 4: 3}, 0.02),
    "short_four_body": ({2: 3, 3: 2, 4: 1}, 0.02),
    "hcp": ({2: 1.45, 3: 1.05, 4: 1.05}, 0.01),
}


def listed():
    return [
        # one updater driven a change at a time, as a Python sampler drives
        # the reference's updater: the smallest calls
        {"name": "updater_binary", "path": "updater", "lattice": "fcc", "species": 2, "clusters": "pairs_triplets",
         "lo": 10, "hi": 10, "changes": 64},
        {"name": "updater_ternary_four_body", "path": "updater", "lattice": "fcc", "species": 3,
         "clusters": "four_body", "lo": 8, "hi": 8, "changes": 32},
        # one chain alone on the device: a sampler object's runMC
        {"name": "one_chain_binary", "path": "chains", "lattice": "fcc", "species": 2, "clusters": "pairs_triplets",
         "lo": 10, "hi": 10, "chains": 1, "ensemble": "canonical", "t_lo": 800.0, "t_hi": 800.0, "sweeps": 40.0,
         "hooks": False},
        # the benchmark's headline: a phase diagram's grid of temperatures and
        # chemical potentials, 500 sweeps each
        {"name": "grid_sgc_binary", "path": "chains", "lattice": "fcc", "species": 2, "clusters": "pairs_triplets",
         "lo": 10, "hi": 10, "chains": 1024, "ensemble": "sgc", "t_lo": 300.0, "t_hi": 1500.0, "sweeps": 500.0,
         "hooks": False},
        # ternary alloys of many compositions in cells of uneven sizes
        {"name": "uneven_ternary", "path": "chains", "lattice": "fcc", "species": 3, "clusters": "four_body",
         "lo": 8, "hi": 16, "chains": 256, "ensemble": "canonical", "t_lo": 300.0, "t_hi": 1500.0, "sweeps": 20.0,
         "hooks": False},
        # one short launch over a job server's mix: binary and ternary,
        # canonical and SGC, 216 to 13824 sites
        {"name": "job_mix", "path": "chains", "lattice": "fcc", "species": 0, "clusters": "jobs", "lo": 6, "hi": 24,
         "chains": 48, "ensemble": "mixed", "t_lo": 300.0, "t_hi": 1500.0, "sweeps": 0.5, "hooks": False},
        # small quaternary cells in the grand-canonical ensemble
        {"name": "sgc_quaternary", "path": "chains", "lattice": "fcc", "species": 4, "clusters": "third_shell",
         "lo": 8, "hi": 8, "chains": 128, "ensemble": "sgc", "t_lo": 300.0, "t_hi": 1500.0, "sweeps": 8.0,
         "hooks": False},
        # a lattice whose neighbours come from its translation table
        {"name": "hcp_ternary", "path": "chains", "lattice": "hcp", "species": 3, "clusters": "hcp", "lo": 6, "hi": 6,
         "chains": 48, "ensemble": "canonical", "t_lo": 300.0, "t_hi": 1500.0, "sweeps": 10.0, "hooks": False},
        # fixed sites and a bias potential on the composition
        {"name": "constrained_sgc", "path": "chains", "lattice": "fcc", "species": 2, "clusters": "pairs_triplets",
         "lo": 8, "hi": 8, "chains": 16, "ensemble": "sgc", "t_lo": 300.0, "t_hi": 1500.0, "sweeps": 20.0,
         "hooks": True},
        # replica exchange on the largest lattices, one sweep and exchange a pass
        {"name": "tempering_quaternary", "path": "tempering", "lattice": "fcc", "species": 4,
         "clusters": "third_shell", "lo": 32, "hi": 32, "chains": 128, "t_lo": 200.0, "t_hi": 2000.0, "cycles": 1},
        # Wang-Landau walkers, one histogram each, flatness tested as they go
        {"name": "walkers_binary", "path": "walkers", "lattice": "fcc", "species": 2, "clusters": "pairs_triplets",
         "lo": 10, "hi": 10, "chains": 64, "bins": 100, "checks": 8, "check_every": 5000},
        # a whole lattice set at once and its correlation functions from scratch
        {"name": "functions_ternary", "path": "functions", "lattice": "fcc", "species": 3, "clusters": "four_body",
         "lo": 24, "hi": 24},
    ]


def _log(rng, lo, hi):
    return math.exp(rng.uniform(math.log(lo), math.log(hi)))


def draw(rng):
    kind = rng.choice(["updater", "functions", "tempering", "walkers"] + ["chains"] * 6)
    case = {"path": kind, "lattice": "fcc"}
    if kind == "updater":
        case["species"], case["clusters"] = rng.choice([(2, "pairs_triplets"), (3, "four_body"), (2, "pairs"),
                                                        (4, "short_four_body")])
        case["lo"] = case["hi"] = rng.randint(6, 16)
        case["changes"] = rng.randint(9, 64)
    elif kind == "functions":
        case["species"], case["clusters"] = rng.choice([(2, "pairs_triplets"), (3, "four_body")])
        case["lo"] = case["hi"] = rng.randint(9, 24)
    elif kind == "tempering":
        case["species"], case["clusters"] = rng.choice([(2, "pairs_triplets"), (3, "four_body"), (4, "third_shell")])
        case["lo"] = case["hi"] = int(_log(rng, 8, 28))
        case["chains"] = int(_log(rng, 8, 100))
        case["t_lo"], case["t_hi"] = rng.choice([(200.0, 2000.0), (300.0, 1200.0)])
        case["cycles"] = rng.choice([1, 3, 17]) if case["lo"] < 16 else 1
    elif kind == "walkers":
        case["species"], case["clusters"] = rng.choice([(2, "pairs_triplets"), (3, "four_body")])
        case["lo"] = case["hi"] = rng.randint(6, 12)
        case["chains"] = int(_log(rng, 4, 200))
        case["bins"] = rng.choice([37, 100, 250])
        case["checks"], case["check_every"] = rng.randint(1, 6), rng.randint(500, 3000)
    else:
        case["ensemble"] = rng.choice(["canonical", "sgc"])
        form = rng.choice(["binary", "binary", "ternary", "ternary", "quaternary", "mix", "hcp", "hooks"])
        case["hooks"] = form == "hooks"
        case["species"], case["clusters"] = {
            "binary": (2, "pairs_triplets"), "hooks": (2, "pairs_triplets"), "ternary": (3, "four_body"),
            "quaternary": (4, rng.choice(["third_shell", "short_four_body"])), "mix": (0, "jobs"),
            "hcp": (3, "hcp")}[form]
        if form == "mix":
            case["ensemble"] = "mixed"
        if form == "hooks":
            case["ensemble"] = "sgc"
        if form == "hcp":
            case["lattice"] = "hcp"
            case["lo"] = case["hi"] = rng.randint(4, 8)
        elif form == "quaternary":
            case["lo"] = case["hi"] = rng.randint(6, 14)
        else:
            case["lo"] = rng.randint(6, 14)
            case["hi"] = rng.randint(case["lo"], 18)
        case["chains"] = int(_log(rng, 1, 40 if form in ("hooks", "hcp") else 1200))
        t_lo = rng.uniform(250.0, 900.0)
        case["t_lo"], case["t_hi"] = round(t_lo, 1), round(rng.uniform(t_lo, 1500.0), 1)
        # moves of all chains, weighted by the work of one: at most a third of
        # the largest listed case's
        per = {2: 1.0, 3: 12.0, 0: 8.0, 4: 40.0}[case["species"]]
        sites = (0.5 * (case["lo"] + case["hi"])) ** 3
        sweeps = min(_log(rng, 0.5, 60.0), 1.5e8 / (per * sites * case["chains"]), 2e5 / (sites * math.sqrt(per)))
        case["sweeps"] = round(max(sweeps, 0.2), 2)
    return case


# ------------------------------------------------------------------ inputs
def _settings(case, species, clusters, size):
    from cemc_amd.crystal import HCPSettings
    from cemc_amd.lattice import FCCSettings, seeded_ecis
    shells, sigma = INTERACTIONS[clusters]
    names = list("ABCD"[:species])
    if case["lattice"] == "hcp":
        st = HCPSettings((size, size, max(4, size - 1)), names, shells)
    else:
        st = FCCSettings(size, names, shells)
    return st, seeded_ecis(st, 2024 + species, sigma)


def _chain_inputs(case, seed):
    """Settings per chain and chain descriptions, made from the seed alone."""
    rng = np.random.Generator(np.random.Philox(seed))
    made, out = {}, []
    n = case["chains"]
    temps = np.geomspace(case.get("t_lo", 1000.0), case.get("t_hi", 1000.0), min(n, 64))
    mus = np.linspace(-0.2, 0.2, 8)
    sizes = np.linspace(case["lo"], case["hi"], n).round().astype(int) if n > 1 else [case["hi"]]
    for c in range(n):
        species = case["species"] or 2 + c % 2
        clusters = case["clusters"] if case["species"] else ("pairs_triplets", "four_body")[c % 2]
        ensemble = case.get("ensemble", "canonical")
        if ensemble == "mixed":
            ensemble = ("canonical", "sgc")[(c // 2) % 2]
        key = (species, int(sizes[c]))
        if key not in made:
            made[key] = _settings(case, species, clusters, int(sizes[c]))
        st, eci = made[key]
        if ensemble == "sgc" or species == 2 or case["path"] != "chains":
            frac = np.full(species, 1.0 / species)
        else:  # canonical multi-component alloys: a random composition each
            frac = np.maximum(rng.dirichlet(np.ones(species)), 0.02)
            frac = frac / frac.sum()
        counts = np.maximum(np.floor(frac * st.n_sites).astype(int), 1)
        counts[0] += st.n_sites - counts.sum()
        occ = rng.permutation(np.repeat(np.arange(species), counts)).astype(np.int8)
        chain = dict(kind=1 if ensemble == "sgc" else 0, temperature=float(temps[c % len(temps)]), occupation=occ,
                     seed=int(rng.integers(1 << 62)), uid=c)
        if chain["kind"]:
            chain["chem_pot"] = {"c1_%d" % d: float(mus[(c // 64 + d) % 8 if n > 64 else (c + d) % 8])
                                 for d in range(species - 1)}
        hooks = None
        if case.get("hooks"):
            # a tenth of the sites fixed, and a parabolic bias on the count of A
            allowed = np.where(rng.random(st.n_sites) < 0.1, 0, 2 ** species - 1).astype(np.uint8)
            x = np.arange(st.n_sites + 1) / st.n_sites
            hooks = dict(allowed=allowed, bias_species=0, bias_table=4.0 * (x - 0.4) ** 2, max_attempts=1000)
        out.append((key, chain, hooks))
    return made, out


def _batch(case, seed):
    from cemc_amd.batch import ChainBatch
    from cemc_amd.model import CEModel
    made, chains = _chain_inputs(case, seed)
    models = {k: CEModel(st, eci) for k, (st, eci) in made.items()}
    batch = ChainBatch([models[k] for k, _, _ in chains], [c for _, c, _ in chains])
    for i, (_, _, hooks) in enumerate(chains):
        if hooks:
            batch.set_hooks(i, **hooks)
    return batch


def _moves(case, n_sites):
    return max(1, int(round(case["sweeps"] * n_sites)))


def _walker_range(e0, bins):
    """The start a third of a bin from an edge, 2 eV to either side."""
    width = 4.0 / bins
    lo = e0 - (bins // 2) * width - width / 3.0
    return lo, lo + 4.0


_KEPT = {}  # one updater per process and kind of lattice, as a program holds one


def _updater_inputs(case, seed):
    st, eci = _settings(case, case["species"], case["clusters"], case["hi"])
    rng = np.random.Generator(np.random.Philox(seed))
    occ = rng.permutation(np.arange(st.n_sites) % case["species"]).astype(np.int8)
    at = occ.copy()
    moves = []
    for _ in range(case.get("changes", 0)):
        i = int(rng.integers(st.n_sites))
        j = int(rng.choice(np.flatnonzero(at != at[i])))
        keep = bool(rng.integers(2))
        moves.append((i, j, int(at[i]), int(at[j]), keep))
        if keep:
            at[i], at[j] = at[j], at[i]
    return st, eci, occ, moves


def prepare(case, seed):
    if case["path"] in ("updater", "functions"):
        from cemc_amd.lattice import SimpleAtoms
        from cemc_amd.updater import PyCEUpdater
        st, eci, occ, moves = _updater_inputs(case, seed)
        key = (case["species"], case["clusters"], case["hi"])
        if key not in _KEPT:
            for other in _KEPT.values():
                other.close()
            _KEPT.clear()
            _KEPT[key] = PyCEUpdater(SimpleAtoms([st.species[v] for v in occ]), st, None, dict(eci))
        names = st.species
        swaps = [([(i, names[a], names[b]), (j, names[b], names[a])], keep) for i, j, a, b, keep in moves]
        return {"path": case["path"], "updater": _KEPT[key], "symbols": [names[v] for v in occ], "swaps": swaps}
    state = {"path": case["path"], "batch": _batch(case, seed)}
    n_sites = state["batch"].n_sites
    if case["path"] == "chains":
        state["moves"] = np.array([_moves(case, int(n)) for n in n_sites], dtype=np.int64)
    elif case["path"] == "tempering":
        from cemc_amd.tempering import ReplicaExchange
        state.update(exchange=ReplicaExchange(state["batch"], seed=seed, uid=1 << 40), cycles=case["cycles"],
                     moves=int(n_sites[0]))
    else:
        for c, e in enumerate(state["batch"].energies()):
            lo, hi = _walker_range(e, case["bins"])
            state["batch"].wl_set(c, case["bins"], lo, hi, 1.0, 1e-8, 0.8, current_bin=case["bins"] // 2)
        state.update(checks=case["checks"], check_every=case["check_every"])
    return state


def _sampled(batch):
    out = batch.stats()
    out["energy"] = batch.energies()
    out["lattice"] = np.concatenate([batch.occupation(c) for c in range(batch.n_chains)])
    return out


def run(state):
    path = state["path"]
    if path in ("updater", "functions"):
        upd = state["updater"]
        upd.set_symbols(state["symbols"])
        if path == "functions":
            return {"cf": upd.get_cf_array(), "energy": upd.get_energy()}
        energies = np.zeros(len(state["swaps"]))
        for k, (changes, keep) in enumerate(state["swaps"]):
            energies[k] = upd.calculate(changes)
            if keep:
                upd.clear_history()
            else:
                upd.undo_changes()
        return {"energies": energies, "cf": upd.get_cf_array(), "lattice": upd.get_occupation()}
    batch = state["batch"]
    if path == "chains":
        batch.run(state["moves"])
        return _sampled(batch)
    if path == "tempering":
        state["exchange"].run(state["cycles"], state["moves"])
        out = _sampled(batch)
        out.update({k: v for k, v in state["exchange"].state().items() if k != "temperatures"})
        return out
    batch.wl_run(state["checks"], state["check_every"])
    walkers = [batch.wl_get(c) for c in range(batch.n_chains)]
    out = {k: np.stack([w[k] for w in walkers]) for k in ("logdos", "hist", "known")}
    out.update({k: np.array([w[k] for w in walkers]) for k in ("f", "current_bin", "n_accept", "n_outside")})
    out["energy"] = batch.energies()
    out["lattice"] = np.concatenate([batch.occupation(c) for c in range(batch.n_chains)])
    return out


# ------------------------------------------------------- cost and tolerance
# sub-clusters that hold a given site
SUBCLUSTERS = {"pairs": 18, "pairs_triplets": 114, "four_body": 494, "third_shell": 1746, "short_four_body": 110,
               "hcp": 50}


def work(case):
    """Lattices and tables once in and out, and one multiply-add per basis
    function, sub-cluster and changed site, which is what the energy change
    of a move (or a correlation function's sum over the lattice) is."""
    def lattice(size):
        return 2 * size * size * max(4, size - 1) if case["lattice"] == "hcp" else size ** 3

    if case["path"] in ("updater", "functions"):
        flips = 2 * case["changes"] if case["path"] == "updater" else lattice(case["hi"])
        return {"bytes": 2.0 * lattice(case["hi"]) + 8.0 * 2 * SUBCLUSTERS[case["clusters"]],
                "flops": 2.0 * flips * (case["species"] - 1) * SUBCLUSTERS[case["clusters"]]}
    n = case["chains"]
    sizes = np.linspace(case["lo"], case["hi"], n).round() if n > 1 else [case["hi"]]
    total = {"bytes": 0.0, "flops": 0.0}
    for c in range(n):
        sites = lattice(float(sizes[c]))
        species = case["species"] or 2 + c % 2
        subs = SUBCLUSTERS[case["clusters"]] if case["species"] else SUBCLUSTERS[("pairs_triplets", "four_body")[c % 2]]
        if case["path"] == "walkers":
            moves = case["checks"] * case["check_every"]
        elif case["path"] == "tempering":
            moves = case["cycles"] * sites
        else:
            moves = case["sweeps"] * sites
        flips = 1 if case.get("ensemble") == "sgc" else 2
        total["bytes"] += 2.0 * sites + 16.0 * subs
        total["flops"] += 2.0 * moves * flips * (species - 1) * subs
    return total


def tolerance(case):
    # The decisions, and with them the lattices and counts, come out the same
    # for every correct evaluation of the energies in 64 bits; energies and
    # sums differ by the order of their additions.
    # Plain numpy and this framework are 1e-15 to 1.5e-14 apart (rel) after
    # 500 to 40000 moves a chain; sums over 500 sweeps grow to some 1e-13, and
    # a single chain's value may lie near zero.
    if case["path"] in ("updater", "functions"):
        return {"rel": 1e-13, "max": 1e-12, "differ": 0.0}
    return {"rel": 1e-12, "max": 1e-10, "differ": 0.0}


# -------------------------------------------------------- plain 64-bit results
class _Plain:
    """A lattice's energy, correlation functions and energy changes from the
    definition (cluster sums of products of basis functions), in numpy."""

    def __init__(self, st, eci, chem_pot=None):
        self.names = sorted(eci)
        eci = {k: v - (chem_pot or {}).get(k, 0.0) for k, v in eci.items()}
        self.eci = eci
        sp = list(st.species)
        self.phi = np.array([[bf[s] for s in sp] for bf in st.basis_functions])
        S = len(sp)
        self.n, self.S = st.n_sites, S
        cols = [int(c) for c in st.trans_cols]
        slot = {c: j for j, c in enumerate(cols)}
        self.rows = np.concatenate([np.asarray(st.trans_table, dtype=np.int64), np.arange(self.n)[:, None]], axis=1)
        self.single = sum(eci["c1_%d" % d] * self.phi[d] for d in range(S - 1))
        self.group = np.zeros(self.n, dtype=int)
        for g, sites in enumerate(st.index_by_trans_symm):
            self.group[list(sites)] = g
        total = {}
        for info in st.cluster_info:
            for name, cl in info.items():
                total[name] = total.get(name, 0) + len(cl["indices"])
        # per group and sub-cluster: members, what each adds to the table
        # index per species id, and the table; per correlation function and
        # group the same table with the function's own weights
        self.records, tables, at = [], [], 0
        self.deco = {cf: [] for cf in self.names}
        for g, info in enumerate(st.cluster_info):
            member, stride, ref_stride, base = [], [], [], []
            per_site = 1.0 / int((self.group == g).sum())
            for name, cl in info.items():
                n = int(cl["size"])
                if n < 2:
                    continue
                w = np.zeros((S,) * n)
                for cf in self.names:
                    if cf.rsplit("_", 1)[0] != name:
                        continue
                    decos = [[int(ch) for ch in cf.rsplit("_", 1)[1]]]
                    for same in cl["equiv_sites"]:
                        grown = []
                        for d in decos:
                            for perm in itertools.permutations([d[p] for p in same]):
                                e = list(d)
                                for p, v in zip(same, perm):
                                    e[p] = v
                                grown.append(e)
                        decos = grown
                    term = np.zeros((S,) * n)
                    for d in decos:
                        t = np.ones(())
                        for v in d:
                            t = np.multiply.outer(t, self.phi[v])
                        term += t / len(decos)
                    term *= per_site / total[name]
                    self.deco[cf].append((at, term.ravel()))
                    w += eci[cf] * n * self.n * term
                strides = [S ** (n - 1 - k) for k in range(n)]
                for sub, order in zip(cl["indices"], cl["order"]):
                    place = {int(who): strides[pos] for pos, who in enumerate(order)}
                    member.append([slot[int(c)] for c in sub] + [len(cols)] * (4 - n))
                    stride.append([place[q + 1] for q in range(n - 1)] + [0] * (4 - n))
                    ref_stride.append(place[0])
                    base.append(at)
                tables.append(w.ravel())
                at += w.size
            self.records.append(tuple(np.array(v) for v in (member, stride, ref_stride, base)))
        self.table = np.concatenate(tables)

    def change(self, occ, i, new):
        """Energy change of setting site i to `new`."""
        member, stride, ref, base = self.records[self.group[i]]
        k = base + (occ[self.rows[i][member]] * stride).sum(axis=1)
        d = self.table[k + int(new) * ref] - self.table[k + int(occ[i]) * ref]
        return float(d.sum() + self.single[new] - self.single[occ[i]])

    def functions(self, occ):
        occ = np.asarray(occ, dtype=np.int64)
        count = np.zeros(self.table.size)
        for g, (member, stride, ref, base) in enumerate(self.records):
            sites = np.flatnonzero(self.group == g)
            for i in range(0, len(sites), 512):
                at = sites[i:i + 512]
                k = base + (occ[self.rows[at][:, member]] * stride).sum(axis=2) + occ[at, None] * ref
                count += np.bincount(k.ravel(), minlength=count.size)
        out = []
        for name in self.names:
            if name.startswith("c0"):
                out.append(1.0)
            elif name.startswith("c1"):
                out.append(float(self.phi[int(name.rsplit("_", 1)[1])][occ].mean()))
            else:
                out.append(sum(float(count[at:at + t.size] @ t) for at, t in self.deco[name]))
        return np.array(out)

    def energy(self, occ):
        return float(self.n * (np.array([self.eci[k] for k in self.names]) @ self.functions(occ)))


def _blocks(seed, uid, counter, n):
    """n Philox4x64-10 blocks; counter: (first move, attempt)."""
    start = (counter[0] + (counter[1] << 64) - 1) % (1 << 256)
    ctr = np.array([(start >> (64 * i)) & ((1 << 64) - 1) for i in range(4)], dtype=np.uint64)
    raw = np.random.Philox(key=np.array([seed, uid], dtype=np.uint64), counter=ctr).random_raw(4 * n)
    return [[int(v) for v in b] for b in raw.reshape(n, 4)]


class _Chain:
    """Proposals of one chain and its lattice."""

    def __init__(self, plain, chain):
        self.p, self.occ, self.kind = plain, chain["occupation"].astype(np.int64), chain["kind"]
        self.key = (chain["seed"], chain["uid"])
        self.present = [s for s in range(plain.S) if (self.occ == s).any()]
        self.where = {s: list(np.flatnonzero(self.occ == s)) for s in self.present}

    def propose(self, w):
        """(changes, tracker slots) of Philox block w."""
        low = w[0] & 0xFFFFFFFF
        if self.kind:
            i = (w[1] * self.p.n) >> 64
            new = (int(self.occ[i]) + 1 + ((low * (self.p.S - 1)) >> 32)) % self.p.S
            return [(i, new)], None
        n = len(self.present)
        ia = ((w[0] >> 32) * n) >> 32
        a, b = self.present[ia], self.present[(ia + 1 + ((low * (n - 1)) >> 32)) % n]
        sa, sb = (w[1] * len(self.where[a])) >> 64, (w[2] * len(self.where[b])) >> 64
        return [(int(self.where[a][sa]), b), (int(self.where[b][sb]), a)], (a, sa, b, sb)

    def change(self, changes):
        """Energy change; the lattice is left changed."""
        de = 0.0
        for i, new in changes:
            de += self.p.change(self.occ, i, new)
            self.occ[i] = new
        return de

    def keep(self, changes, slots):
        if slots:
            a, sa, b, sb = slots
            self.where[a][sa], self.where[b][sb] = changes[1][0], changes[0][0]


def _metropolis(plain, chain, hooks, moves):
    ch = _Chain(plain, chain)
    kt = KB * chain["temperature"]
    bias = hooks["bias_table"] if hooks else None
    count = int((ch.occ == 0).sum())
    e = plain.energy(ch.occ) + (bias[count] if hooks else 0.0)
    accepted, s1, s2 = 0, [], []
    for t, w in enumerate(_blocks(*ch.key, (0, 0), moves)):
        changes, slots = ch.propose(w)
        attempt = 0
        while hooks and not all((int(hooks["allowed"][i]) >> new) & 1 for i, new in changes):
            attempt += 1
            w = _blocks(*ch.key, (t, attempt), 1)[0]
            changes, slots = ch.propose(w)
        old = [(i, int(ch.occ[i])) for i, _ in changes]
        de, dn = ch.change(changes), 0
        if hooks:
            dn = sum((new == 0) - (o == 0) for (_, new), (_, o) in zip(changes, old))
            de += bias[count + dn] - bias[count]
        if de < 0.0 or (w[3] >> 11) * 2.0 ** -53 <= math.exp(-de / kt):
            e, accepted, count = e + de, accepted + 1, count + dn
            ch.keep(changes, slots)
        else:
            for i, o in reversed(old):
                ch.occ[i] = o
        s1.append(e)
        s2.append(e * e)
    return moves, accepted, math.fsum(s1), math.fsum(s2), e, ch.occ.astype(np.int8)


def _walker(plain, chain, case):
    ch = _Chain(plain, chain)
    e = plain.energy(ch.occ)
    bins = case["bins"]
    lo, hi = _walker_range(e, bins)
    g, hist, known = np.zeros(bins), np.zeros(bins, dtype=np.int32), np.zeros(bins, dtype=np.uint8)
    f, cur, first, accepted, outside = 1.0, bins // 2, True, 0, 0
    blocks = iter(_blocks(*ch.key, (0, 0), case["checks"] * case["check_every"]))
    for _ in range(case["checks"]):
        for _ in range(case["check_every"]):
            w = next(blocks)
            changes, slots = ch.propose(w)
            old = [(i, int(ch.occ[i])) for i, _ in changes]
            en = e + ch.change(changes)
            at = math.trunc((en - lo) * bins / (hi - lo)) if en >= lo or (lo - en) * bins < hi - lo else -1
            take = False
            if 0 <= at < bins:
                diff = g[cur] - g[at]
                take = first or (w[3] >> 11) * 2.0 ** -53 < (1.0 if diff > 0 else math.exp(diff))
            if take:
                e, cur, first, accepted = en, at, False, accepted + 1
                ch.keep(changes, slots)
            else:
                for i, o in reversed(old):
                    ch.occ[i] = o
            if not 0 <= at < bins:
                outside += 1
                if first or at <= bins:
                    continue
            g[cur] += f
            hist[cur] += 1
            known[cur] = 1
        seen = hist[known > 0]
        if len(seen) and seen.min() > 0.8 * seen.mean():
            f /= 2.0
            hist[:] = 0
    return g, hist, known, f, cur, accepted, outside, e, ch.occ.astype(np.int8)


def exact(case, seed):
    if case["path"] in ("updater", "functions"):
        st, eci, occ, moves = _updater_inputs(case, seed)
        plain = _Plain(st, eci)
        occ = occ.astype(np.int64)
        if case["path"] == "functions":
            return {"cf": plain.functions(occ), "energy": plain.energy(occ)}
        e = plain.energy(occ)
        energies = []
        for i, j, a, b, keep in moves:
            de = plain.change(occ, i, b)
            occ[i] = b
            de += plain.change(occ, j, a)
            occ[j] = a
            energies.append(e + de)
            if keep:
                e += de
            else:
                occ[i], occ[j] = a, b
        return {"energies": np.array(energies), "cf": plain.functions(occ), "lattice": occ.astype(np.int8)}
    if case["path"] == "tempering":
        return None
    n = case["chains"]
    sizes = np.linspace(case["lo"], case["hi"], n).round() if n > 1 else [case["hi"]]
    moves = [case["checks"] * case["check_every"] if case["path"] == "walkers" else case["sweeps"] * s ** 3
             for s in sizes]
    cost = {2: 6e-5, 3: 9e-5, 0: 9e-5, 4: 2e-4}[case["species"]]
    if cost * sum(moves) > 18.0:
        return None
    made, chains = _chain_inputs(case, seed)
    got, plains = [], {}
    for key, chain, hooks in chains:
        mu = chain.get("chem_pot") or {}
        of = (key, tuple(sorted(mu.items())))
        if of not in plains:
            plains[of] = _Plain(*made[key], mu)
        if case["path"] == "walkers":
            got.append(_walker(plains[of], chain, case))
        else:
            got.append(_metropolis(plains[of], chain, hooks, _moves(case, made[key][0].n_sites)))
    if case["path"] == "walkers":
        g, hist, known, f, cur, acc, outside, e, occ = zip(*got)
        return {"logdos": np.stack(g), "hist": np.stack(hist), "known": np.stack(known), "f": np.array(f),
                "current_bin": np.array(cur), "n_accept": np.array(acc), "n_outside": np.array(outside),
                "energy": np.array(e), "lattice": np.concatenate(occ)}
    made_, acc, s1, s2, e, occ = zip(*got)
    return {"moves": np.array(made_), "accepted": np.array(acc), "sum_e": np.array(s1), "sum_e2": np.array(s2),
            "energy": np.array(e), "lattice": np.concatenate(occ)}

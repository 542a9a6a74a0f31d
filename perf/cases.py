"""Measured workloads of the framework, through the Engine calls a user's program makes.

The listed cases are the work this library is run for, over its range of sizes:
the semi-grand canonical T x mu grid, a single canonical chain, canonical batches
of a binary, a ternary and a quaternary expansion, a ragged supercell, the N-fold
way, the learned proposal and its training, and the per-proposal and
whole-configuration evaluations (energy changes, correlations).  ``draw`` gives
other sizes, chain counts and options of the same workloads.

A case is a dict of plain values; ``work`` (its "kind") says which call it is:

  sgc / canonical   Engine.run_passes on loaded, equilibrated chains, samples read
  run               load_chains + run_passes + read_samples + read_state: one
                    whole run from host states to host results
  nfold             Engine.nfold_run_moments on loaded, equilibrated chains
  learned           Engine.run_passes with the learned proposal
  delta             Engine.delta_energy_batch on loaded chains
  corr              load_chains + correlations + energy of every chain
  train             Engine.mlp_train from given parameters
  gradients         Engine.mlp_gradients on given rows
"""
from __future__ import annotations

import functools

import numpy as np

from casmcode_clexmonte_amd.engine import Engine
from casmcode_clexmonte_amd.system import FlatCE, Supercell
from casmcode_clexmonte_amd.workloads import (bcc_quaternary_ce, fcc_binary_ce, fcc_ordering_ce, hcp_ternary_ce,
                                              l12_occupation, random_mlp_params)

_CE = {"fcc": fcc_binary_ce, "fcc_ordering": fcc_ordering_ce, "hcp": hcp_ternary_ce, "bcc": bcc_quaternary_ce}
# occupant fractions of the canonical workloads
_X = {"fcc": (0.5, 0.5), "fcc_ordering": (0.75, 0.25), "hcp": (0.4, 0.3, 0.3), "bcc": (0.25, 0.25, 0.25, 0.25)}
KB = 8.6173303e-05


def listed():
    return [
        # the headline grid: FCC binary 24^3, 16 T x 16 mu, 20 sampled passes per call
        dict(name="sgc_fcc24_grid", kind="sgc", ce="fcc", dims="24x24x24", chains=256, T0=200.0, T1=1500.0,
             mu=0.3, passes=20, period=1),
        # one small canonical chain at 600 K, a whole short run: the latency-bound end
        dict(name="run_fcc12_chain", kind="run", ce="fcc", dims="12x12x12", chains=1, T0=600.0, T1=600.0,
             ensemble="canonical", passes=100, period=1, rounds=2, pairs=8),
        # canonical batch around the L1_2 ordering temperature, automatic rounds
        dict(name="canonical_fcc32_batch", kind="canonical", ce="fcc_ordering", dims="32x32x32", chains=128,
             T0=119.0, T1=221.0, passes=10, period=1, rounds=0, pairs=4),
        # ternary semi-grand canonical chains on a supercell that no periodic colouring fits
        dict(name="sgc_hcp_ragged", kind="sgc", ce="hcp", dims="11x9x7", chains=64, T0=600.0, T1=1800.0, mu=0.2,
             passes=10, period=1),
        # canonical ternary HCP chains on uneven supercells, a whole run from host states
        dict(name="run_hcp_uneven", kind="run", ce="hcp", dims="16x16x12,24x24x16,36x36x24", chains=24, T0=600.0,
             T1=1800.0, ensemble="canonical", passes=8, period=1, rounds=0, pairs=4),
        # the largest chains: quaternary BCC 64^3, equiatomic
        dict(name="canonical_bcc64", kind="canonical", ce="bcc", dims="64x64x64", chains=32, T0=300.0, T1=2000.0,
             passes=8, period=1, rounds=2, pairs=1),
        # rejection-free sampling at low temperature
        dict(name="nfold_fcc24", kind="nfold", ce="fcc", dims="24x24x24", chains=256, T0=200.0, T1=400.0, mu=0.3,
             events=1000, block=100),
        # the learned proposal on the ordering workload
        dict(name="learned_fcc32", kind="learned", ce="fcc_ordering", dims="32x32x32", chains=128, T0=119.0,
             T1=221.0, passes=4, period=1, proposal="learned", rounds=16, pairs=4),
        # one proposed swap (the calculators' occ_delta_per_supercell)
        dict(name="delta_fcc12_one", kind="delta", ce="fcc", dims="12x12x12", chains=1, n=1, sites=2, chem=False),
        # a large batch of proposed swaps over many chains
        dict(name="delta_bcc32_batch", kind="delta", ce="bcc", dims="32x32x32", chains=16, n=65536, sites=2,
             chem=False),
        # states loaded, and every correlation read (the corr.formation_energy sampler)
        dict(name="corr_bcc32", kind="corr", ce="bcc", dims="32x32x32", chains=8),
        # training of the proposal network on the chains' configurations
        dict(name="train_fcc24", kind="train", ce="fcc_ordering", dims="24x24x24", chains=128, T0=119.0, T1=221.0,
             n=512, steps=10),
    ]


def draw(rng):
    """One more case of the listed workloads: another size, chain count or option."""
    def log(lo, hi):
        return max(lo, min(hi, int(round(lo * (hi / lo) ** rng.random()))))

    def dims(lo, hi):
        return "%dx%dx%d" % tuple(rng.randint(lo, hi) for _ in range(3))

    kind = rng.choice(["sgc", "sgc", "canonical", "canonical", "run", "nfold", "learned", "delta", "delta", "corr",
                       "train", "gradients"])
    T0 = float(rng.randint(300, 900))
    T1 = T0 + float(rng.randint(100, 900))
    if kind == "sgc":
        ce = rng.choice(["fcc", "fcc", "hcp", "bcc"])
        m = rng.choice([2, 3])  # divisors the periodic colourings use; 1 in 4 cases has none
        d = dims(6, 10) if rng.random() < 0.25 else "x".join(str(m * 2 * rng.randint(2, 5 if m == 2 else 4))
                                                               for _ in range(3))
        return dict(kind=kind, ce=ce, dims=d, chains=log(1, 300), T0=T0, T1=T1, mu=rng.choice([0.0, 0.1, 0.3]),
                    passes=log(1, 40), period=rng.choice([1, 1, 5]))
    if kind == "canonical":
        ce = rng.choice(["fcc", "hcp", "bcc"])
        d = "x".join(str(4 * rng.randint(2, 7)) for _ in range(3))
        return dict(kind=kind, ce=ce, dims=d, chains=log(1, 128), T0=T0, T1=T1, passes=log(1, 12),
                    period=rng.choice([1, 1, 4]), rounds=rng.choice([0, 0, 1, 2]), pairs=rng.randint(1, 4))
    if kind == "run":
        ce = rng.choice(["fcc", "hcp"])
        n = rng.choice([1, 2])
        d = ",".join("x".join(str(4 * rng.randint(2, 5)) for _ in range(3)) for _ in range(n))
        ens = rng.choice(["canonical", "semigrand_canonical"])
        return dict(kind=kind, ce=ce, dims=d, chains=log(2, 32), T0=T0, T1=T1, ensemble=ens, passes=log(2, 50),
                    period=rng.choice([1, 1, 2]), rounds=rng.choice([0, 2]), pairs=rng.randint(0, 4))
    if kind == "nfold":
        ce = rng.choice(["fcc", "fcc", "hcp"])
        block = rng.choice([50, 100, 250])
        return dict(kind=kind, ce=ce, dims=dims(8, 20), chains=log(1, 256), T0=T0, T1=T1,
                    mu=rng.choice([0.0, 0.1, 0.3]), events=block * rng.randint(1, 4), block=block)
    if kind == "learned":
        d = "x".join(str(4 * rng.randint(2, 7)) for _ in range(3))
        return dict(kind=kind, ce="fcc_ordering", dims=d, chains=log(1, 96), T0=130.0, T1=float(rng.randint(150, 400)),
                    passes=log(1, 4), period=1, proposal=rng.choice(["learned", "informed", "grouped_uniform"]),
                    rounds=rng.choice([8, 16]), pairs=rng.randint(1, 4))
    if kind == "delta":
        return dict(kind=kind, ce=rng.choice(["fcc", "hcp", "bcc"]), dims=dims(8, 24), chains=log(1, 16),
                    n=log(1, 60000), sites=rng.randint(1, 4), chem=rng.random() < 0.5)
    if kind == "corr":
        return dict(kind=kind, ce=rng.choice(["fcc", "hcp", "bcc"]), dims=dims(8, 26), chains=log(1, 8))
    if kind == "train":
        return dict(kind=kind, ce="fcc_ordering", dims="16x16x16", chains=log(4, 64), T0=130.0, T1=300.0,
                    n=log(40, 900), steps=rng.randint(1, 8))
    return dict(kind=kind, ce="fcc_ordering", n=log(100, 60000))


# --- systems and inputs --------------------------------------------------------------
@functools.lru_cache(maxsize=None)
def _flat(ce):
    return FlatCE(_CE[ce]())


def _dims(case):
    return [tuple(int(v) for v in d.split("x")) for d in case["dims"].split(",")]


def _supercells(case):
    flat = _flat(case["ce"])
    shapes = [Supercell(flat.ce.prim, d) for d in _dims(case)]
    return [shapes[c % len(shapes)] for c in range(case["chains"])]


@functools.lru_cache(maxsize=None)
def _ordered(dims):
    return l12_occupation(Supercell(_flat("fcc_ordering").ce.prim, dims))


def _occupations(case, seed):
    """Random occupations at the workload's composition (L1_2 below the ordering
    temperature of the ordering workload, where the supercell holds it)."""
    rng = np.random.default_rng(seed)
    temps = _temperatures(case)
    out = []
    for c, sc in enumerate(_supercells(case)):
        if case["ce"] == "fcc_ordering" and temps[c] < 170.0 and all(d % 2 == 0 for d in sc.dims):
            out.append(_ordered(tuple(sc.dims)))
            continue
        counts = [int(round(x * sc.n_sites)) for x in _X[case["ce"]][:-1]]
        occ = np.repeat(np.arange(len(counts) + 1, dtype=np.int8), counts + [sc.n_sites - sum(counts)])
        out.append(rng.permutation(occ))
    return out


def _temperatures(case):
    n = case["chains"]
    return np.linspace(case.get("T0", 600.0), case.get("T1", 600.0), n) if n > 1 else np.array([case.get("T0", 600.0)])


def _chem(case, seed):
    """Occupant weights of every chain: mu over a grid on the second occupant."""
    if "mu" not in case and not case.get("chem") and case.get("ensemble") != "semigrand_canonical":
        return None
    flat = _flat(case["ce"])
    mu = case.get("mu", 0.1)
    w = np.zeros((case["chains"], flat.n_sublat, flat.n_occ_max))
    grid = np.linspace(-mu, mu, 16)
    for c in range(case["chains"]):
        w[c, :, 1] = grid[c % 16]
        if flat.n_occ_max > 2:
            w[c, :, 2] = 0.5 * grid[(c // 16) % 16]
    return w


def _seeds(case, seed):
    return (np.uint64(seed) << np.uint64(20)) + np.arange(case["chains"], dtype=np.uint64)


def _proposals(case, seed):
    """Proposed changes: swaps of two different occupants (two sites), else
    every site to another occupant."""
    rng = np.random.default_rng(seed + 1)
    occ = np.stack(_occupations(case, seed)).astype(np.int32)
    n, m, n_occ = case["n"], case["sites"], int(_flat(case["ce"]).n_occ_max)
    chain = rng.integers(0, case["chains"], n).astype(np.int32)
    sites = rng.integers(0, occ.shape[1], (n, m)).astype(np.int32)
    old = occ[chain[:, None], sites]
    if m == 2:
        while (same := old[:, 0] == old[:, 1]).any():
            sites[same, 1] = rng.integers(0, occ.shape[1], int(same.sum()))
            old = occ[chain[:, None], sites]
        return chain, sites, np.ascontiguousarray(old[:, ::-1])
    return chain, sites, ((old + rng.integers(1, n_occ, (n, m))) % n_occ).astype(np.int32)


def _engine(case):
    """A handle with the case's supercells; returns it and the chains' supercell ids."""
    flat = _flat(case["ce"])
    eng = Engine(flat, device=0)
    ids = {}
    for k, d in enumerate(_dims(case)):
        if d not in ids:
            ids[d] = eng.add_supercell(Supercell(flat.ce.prim, d), n_pair_phases=case.get("pairs", 0), seed=k)
    return eng, [ids[tuple(sc.dims)] for sc in _supercells(case)]


@functools.lru_cache(maxsize=4)
def _kept_engine(key):
    """The handle that a program running one state after another keeps."""
    return _engine(dict(key))


def _load(eng, ids, case, seed):
    eng.load_chains(ids, _occupations(case, seed), _temperatures(case), _seeds(case, seed), chem=_chem(case, seed))


def prepare(case, seed):
    kind = case["kind"]
    if kind in ("run", "corr"):
        eng, ids = _kept_engine(tuple(sorted((k, v) for k, v in case.items() if k != "name")))
        return dict(case=case, eng=eng, args=(ids, _occupations(case, seed), _temperatures(case),
                                              _seeds(case, seed), _chem(case, seed)))
    if kind == "gradients":
        eng = Engine(_flat(case["ce"]), device=0)
        rng = np.random.default_rng(seed)
        n_env = eng.mlp_info()[0]
        eng.mlp_set_params(random_mlp_params(seed % 1000, n_env))
        X = np.zeros((case["n"], 48), np.int8)
        X[:, :n_env] = rng.choice(np.array([-1, 1], np.int8), (case["n"], n_env))
        y = rng.random(case["n"]).astype(np.float32)
        t = rng.uniform(2.0, 10.0, case["n"]).astype(np.float32)
        return dict(case=case, eng=eng, X=X, y=y, t=t, params=random_mlp_params(seed % 1000, n_env))
    eng, ids = _engine(case)
    _load(eng, ids, case, seed)
    st = dict(case=case, eng=eng)
    if kind == "delta":
        st["chain"], st["sites"], st["new"] = _proposals(case, seed)
        return st
    # equilibration, as a program does before it samples
    if kind == "canonical":
        eng.run_passes("canonical", 4, 4, case["rounds"])
    elif kind in ("sgc", "nfold"):
        eng.run_passes("semigrand_canonical", 20, 20)
    elif kind == "learned":
        eng.run_passes("canonical", 4, 4, 0)
        eng.mlp_set_params(random_mlp_params(seed % 1000, eng.mlp_info()[0]))
        eng.set_proposal(case["proposal"], rounds_per_group=case["rounds"])
    elif kind == "train":
        st["params"] = random_mlp_params(seed % 1000, eng.mlp_info()[0])
        st["seed"] = seed % (1 << 31)
    return st


def run(s):
    case, eng = s["case"], s["eng"]
    kind = case["kind"]
    if kind == "sgc" or kind == "canonical" or kind == "learned":
        eng.clear_samples()
        eng.run_passes("semigrand_canonical" if kind == "sgc" else "canonical", case["passes"], case["period"],
                       canonical_rounds=case.get("rounds", 1) if kind == "canonical" else 0)
        E, counts = eng.read_samples()
        return {"E": E, "counts": counts}
    if kind == "run":
        eng.load_chains(*s["args"][:4], chem=s["args"][4])
        eng.run_passes(case["ensemble"], case["passes"], case["period"], canonical_rounds=case["rounds"])
        E, counts = eng.read_samples()
        states = [eng.read_state(c) for c in range(case["chains"])]
        return {"E": E, "counts": counts, "occ": np.concatenate([x["occ"] for x in states]),
                "E_end": np.array([x["E"] for x in states]), "attempts": np.array([x["n_attempt"] for x in states]),
                "accepts": np.array([x["n_accept"] for x in states])}
    if kind == "nfold":
        return eng.nfold_run_moments(case["events"], case["block"])
    if kind == "delta":
        return eng.delta_energy_batch(s["chain"], s["sites"], s["new"], include_chem=case["chem"])
    if kind == "corr":
        eng.load_chains(*s["args"][:4], chem=s["args"][4])
        return {"corr": np.stack([eng.correlations(c) for c in range(case["chains"])]),
                "E": np.array([eng.read_state(c)["E"] for c in range(case["chains"])])}
    if kind == "train":
        eng.mlp_set_params(s["params"])
        loss = eng.mlp_train(case["n"], case["steps"], lr=3e-3, seed=s["seed"])
        return {"loss": loss, "params": eng.mlp_get_params()}
    grad, loss = eng.mlp_gradients(s["X"], s["y"], s["t"])
    return {"grad": grad, "loss": loss}


# --- what a pass cannot do without ----------------------------------------------------
def _ops_per_site(ce):
    """Cluster terms of one site: one operation per other site of every cluster
    that holds it and one per cluster and site function."""
    flat = _flat(ce)
    nf = 1 if flat.binary else flat.n_func_max
    n_var = max(1, sum(1 for n in flat.n_occ if n >= 2))
    return (int(np.sum(flat.entry_k)) + nf * flat.n_entries) / n_var


def work(case):
    kind = case["kind"]
    if kind in ("train", "gradients"):
        n = case["n"] * case.get("chains", 1)
        steps = case.get("steps", 1)
        return {"bytes": n * 57.0 + 4 * 3201 * 2, "flops": steps * 3 * 2.0 * n * 64 * 43}
    n_sites = sum(sc.n_sites for sc in _supercells(case))
    ops = _ops_per_site(case["ce"])
    if kind == "delta":
        # the proposal, its energy and one byte per neighbour
        nb = ops / 2
        return {"bytes": case["n"] * (8.0 + case["sites"] * (8.0 + nb)), "flops": case["n"] * case["sites"] * ops}
    if kind == "corr":
        # each cluster of the supercell once per function
        flat = _flat(case["ce"])
        per_cell = float(np.sum(np.asarray(flat.orbit_mult) * (np.asarray(flat.orbit_nfunc) + np.asarray(flat.orbit_k))))
        cells = sum(sc.n_cells for sc in _supercells(case))
        return {"bytes": n_sites + 8.0 * case["chains"] * (flat.n_corr + 1), "flops": cells * per_cell}
    if kind == "nfold":
        flat = _flat(case["ce"])
        nb = len({tuple(x) for x in np.asarray(flat.entry_sites).reshape(-1, 4).tolist()}) + 1
        return {"bytes": 2.0 * n_sites + 8.0 * 21 * case["chains"] * (case["events"] // case["block"]),
                "flops": (n_sites + case["chains"] * case["events"] * float(nb)) * ops}
    samples = case["chains"] * (case["passes"] // case["period"])
    return {"bytes": 2.0 * n_sites + 24.0 * samples, "flops": case["passes"] * n_sites * ops}


# --- the same in 64 bits ---------------------------------------------------------------
def _entry_values(flat, b, dims, cell, occ_of):
    """Flower sums G[f] (FP64) of sites on sublattice b in cells `cell` [n, 3];
    occ_of(linear site index [n]) gives the occupants."""
    n_cells = dims[0] * dims[1] * dims[2]
    nf = int(flat.n_occ[b]) - 1
    G = np.zeros((len(cell), nf))
    es = np.asarray(flat.entry_sites).reshape(-1, 4)
    tab = np.asarray(flat.flower_tables, float)
    for e in range(int(flat.flower_begin[b]), int(flat.flower_begin[b + 1])):
        idx, mul = np.zeros(len(cell), np.int64), 1
        for q in range(int(flat.entry_site_begin[e]), int(flat.entry_site_begin[e + 1])):
            bq, di, dj, dk = (int(v) for v in es[q])
            i, j, k = (cell[:, 0] + di) % dims[0], (cell[:, 1] + dj) % dims[1], (cell[:, 2] + dk) % dims[2]
            idx += occ_of(bq * n_cells + i + dims[0] * (j + dims[1] * k)) * mul
            mul *= int(flat.n_occ[bq])
        G += tab[int(flat.entry_table[e]) + idx[:, None] * nf + np.arange(nf)]
    return G


def _exact_delta(case, seed):
    flat, dims = _flat(case["ce"]), _dims(case)[0]
    n_cells = dims[0] * dims[1] * dims[2]
    occ = np.stack(_occupations(case, seed)).astype(np.int64)
    chain, sites, new = (x.astype(np.int64) for x in _proposals(case, seed))
    n, m = sites.shape
    chem = _chem(case, seed)
    sf = np.asarray(flat.site_func, float).reshape(flat.n_sublat, flat.n_func_max, flat.n_occ_max)
    dE = np.zeros(n)
    for i in range(m):
        for b in range(flat.n_sublat):
            sel = np.nonzero(sites[:, i] // n_cells == b)[0]
            if len(sel) == 0:
                continue

            def occ_of(l, sel=sel, i=i):
                v = occ[chain[sel], l]
                for j in range(i):
                    v = np.where(sites[sel, j] == l, new[sel, j], v)
                return v

            c = sites[sel, i] % n_cells
            cell = np.stack([c % dims[0], (c // dims[0]) % dims[1], c // (dims[0] * dims[1])], axis=1)
            o, w = occ_of(sites[sel, i]), new[sel, i]
            G = _entry_values(flat, b, dims, cell, occ_of)
            for f in range(G.shape[1]):
                dE[sel] += (sf[b, f, w] - sf[b, f, o]) * G[:, f]
            if case["chem"]:
                dE[sel] -= chem[chain[sel], b, w] - chem[chain[sel], b, o]
    return dE


def _exact_corr(case, seed):
    flat, dims = _flat(case["ce"]), _dims(case)[0]
    n_cells = dims[0] * dims[1] * dims[2]
    occ = np.stack(_occupations(case, seed)).astype(np.int64)
    es = np.asarray(flat.corr_elem_sites).reshape(-1, 4)
    tab = np.asarray(flat.orbit_tables, float)
    grid = occ.reshape(len(occ), flat.n_sublat, dims[2], dims[1], dims[0])
    corr = np.zeros((len(occ), flat.n_corr))
    for a in range(flat.n_orbits):
        k, nf = int(flat.orbit_k[a]), int(flat.orbit_nfunc[a])
        if nf == 0:
            continue
        n_elem = int(flat.corr_orbit_begin[a + 1] - flat.corr_orbit_begin[a])
        first = int(flat.corr_elem_begin[a])
        hist = None
        for e in range(n_elem):
            tau, mul = np.zeros((len(occ), n_cells), np.int64), 1
            for q in range(k):
                b, di, dj, dk = (int(v) for v in es[first + e * k + q])
                tau += np.roll(grid[:, b], (-dk, -dj, -di), (1, 2, 3)).reshape(len(occ), -1) * mul
                mul *= int(flat.n_occ[b])
            h = np.stack([np.bincount(t, minlength=mul) for t in tau])
            hist = h if hist is None else hist + h
        T = tab[int(flat.orbit_table_offset[a]):][:hist.shape[1] * nf].reshape(-1, nf)
        f0 = int(flat.orbit_func_begin[a])
        corr[:, f0:f0 + nf] = hist @ T / float(flat.orbit_mult[a])
    return {"corr": corr, "E": corr @ np.asarray(flat.eci, float)}


def _exact_gradients(case, seed):
    rng = np.random.default_rng(seed)
    n_env = 42  # the sites of the three shortest FCC pair shells: 12 + 6 + 24
    p = np.asarray(random_mlp_params(seed % 1000, n_env), float)
    W1, b1, W2, b2 = p[:3072].reshape(64, 48)[:, :n_env], p[3072:3136], p[3136:3200], p[3200]
    X = rng.choice(np.array([-1, 1], np.int8), (case["n"], n_env)).astype(float)
    y = rng.random(case["n"]).astype(np.float32).astype(float)
    t = rng.uniform(2.0, 10.0, case["n"]).astype(np.float32).astype(float)
    H = X @ W1.T + b1
    A = np.maximum(H, 0.0)
    logit = t * (A @ W2 + b2)
    loss = np.mean(np.logaddexp(0.0, logit) - y * logit)
    dl = t * (1.0 / (1.0 + np.exp(-logit)) - y) / case["n"]
    D = dl[:, None] * W2 * (H > 0)
    g = np.zeros(3201)
    g[:3072].reshape(64, 48)[:, :n_env] = D.T @ X
    g[3072:3136] = D.sum(0)
    g[3136:3200] = A.T @ dl
    g[3200] = dl.sum()
    return {"grad": g, "loss": float(loss)}


def exact(case, seed):
    if case["kind"] == "delta":
        return _exact_delta(case, seed)
    if case["kind"] == "corr":
        return _exact_corr(case, seed)
    if case["kind"] == "gradients":
        return _exact_gradients(case, seed)
    return None

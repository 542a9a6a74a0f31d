"""Correlations by every route: counters in LDS and correlations in one block,
counters in LDS and a second kernel, counters in global memory (an orbit of
eight quaternary sites, 65,536 decorations), several slices of chains (more
than 256 MiB of counters), clusters of more than four sites, and offsets beyond
one period.  All routes form the same sum, so a chain's correlations and energy
are the same bit for bit whatever is loaded beside it.  Against the FP64
oracle: exact counts, one rounded FP64 sum, 1e-12 of the largest value."""
import copy

import numpy as np
import pytest

import oracle as O
from casmcode_clexmonte_amd.engine import Engine
from casmcode_clexmonte_amd.system import FlatCE, Supercell
from casmcode_clexmonte_amd.workloads import bcc_quaternary_ce, fcc_binary_ce, hcp_ternary_ce

pytestmark = pytest.mark.gpu


def _with_orbit(flat, sites, n_func, seed=0):
    """A copy of the expansion with one orbit more: a cluster of `sites` and
    n_func functions of random decoration values, not in the energy."""
    f = copy.copy(flat)
    rng = np.random.default_rng(seed)
    n_tau = int(np.prod([int(flat.n_occ[s[0]]) for s in sites])) if n_func else 0
    f.n_orbits, f.n_corr = flat.n_orbits + 1, flat.n_corr + n_func
    f.orbit_k = np.append(flat.orbit_k, len(sites))
    f.orbit_mult = np.append(flat.orbit_mult, 1)
    f.orbit_nfunc = np.append(flat.orbit_nfunc, n_func)
    f.orbit_func_begin = np.append(np.asarray(flat.orbit_func_begin)[:flat.n_orbits], [flat.n_corr, f.n_corr])
    f.corr_orbit_begin = np.append(flat.corr_orbit_begin, flat.corr_orbit_begin[-1] + 1)
    elem = np.asarray(flat.corr_elem_sites).reshape(-1, 4)
    f.corr_elem_begin = np.append(np.asarray(flat.corr_elem_begin)[:flat.n_orbits], [len(elem), len(elem) + len(sites)])
    f.corr_elem_sites = np.concatenate([elem, np.array(sites, dtype=elem.dtype)])
    f.orbit_table_offset = np.append(np.asarray(flat.orbit_table_offset)[:flat.n_orbits],
                                     [flat.orbit_tables.size] * 2)
    f.orbit_tables = np.append(flat.orbit_tables, rng.normal(0, 1, n_tau * n_func))
    f.eci = np.append(flat.eci, np.zeros(n_func))
    return f


def _loaded(flat, shapes, seed=3):
    eng = Engine(flat)
    scs = [Supercell(flat.ce.prim, d) for d in shapes]
    ids = {d: eng.add_supercell(Supercell(flat.ce.prim, d), n_pair_phases=0) for d in dict.fromkeys(shapes)}
    occs = [np.random.default_rng(seed + c).integers(0, flat.n_occ_max, sc.n_sites).astype(np.int8)
            for c, sc in enumerate(scs)]
    eng.load_chains([ids[d] for d in shapes], occs, [900.0] * len(shapes), list(range(len(shapes))))
    return eng, occs


@pytest.mark.parametrize("ce,small,large", [(fcc_binary_ce, (6, 6, 6), (20, 20, 20)), (hcp_ternary_ce, (4, 5, 4), (14, 12, 12)),
                                            (bcc_quaternary_ce, (4, 4, 5), (14, 14, 14))])
def test_correlations_do_not_depend_on_the_chains_beside(ce, small, large):
    print(f"[case] correlations beside others {ce.__name__}", flush=True)
    flat = FlatCE(ce())
    got = []
    for shapes in ([small, small], [small, small, large]):
        eng, _ = _loaded(flat, shapes)
        got.append([(eng.read_state(c)["E"], eng.correlations(c)) for c in range(2)])
        drift = eng.reanchor_energies()
        assert drift == 0.0
        eng.close()
    for (Ea, ca), (Eb, cb) in zip(*got):
        assert Ea == Eb and np.array_equal(ca, cb)


CLUSTERS = {"eight sites": [(0, 0, 0, 0), (0, 1, 0, 0), (0, 0, 1, 0), (0, 0, 0, 1), (0, 1, 1, 0), (0, 0, 1, 1), (0, 1, 0, 1), (0, 1, 1, 1)],
            "five sites": [(0, 0, 0, 0), (0, 2, 0, 0), (0, 0, 2, 0), (0, -1, 0, 1), (0, 1, 1, 0)],
            "far sites": [(0, 0, 0, 0), (0, 9, -7, 11)]}


@pytest.mark.parametrize("cluster,dims,chains", [("eight sites", (3, 3, 3), 600), ("eight sites", (16, 16, 17), 2),
                                                 ("five sites", (4, 5, 6), 2), ("five sites", (16, 17, 16), 2),
                                                 ("far sites", (4, 5, 6), 2)])
def test_large_clusters(cluster, dims, chains):
    print(f"[case] correlations of {cluster}, {chains} chains of {dims}", flush=True)
    base = FlatCE(bcc_quaternary_ce())
    flat = _with_orbit(base, CLUSTERS[cluster], 2)
    eng, occs = _loaded(flat, [dims] * chains)
    osys = O.OracleSystem(flat, dims)
    plain, _ = _loaded(base, [dims] * chains)
    for c in sorted({0, 1, chains // 2, chains - 1}):
        ref, got = osys.corr(occs[c]), eng.correlations(c)
        assert np.abs(got - ref).max() <= 1e-12 * np.abs(ref).max()
        assert np.array_equal(got[:base.n_corr], plain.correlations(c))
        E = float(flat.eci @ ref)
        assert abs(eng.read_state(c)["E"] - E) <= 1e-9 * max(1.0, abs(E))
    eng.close()
    plain.close()


def test_orbits_without_functions_are_not_counted():
    print("[case] an orbit of 20 sites without functions", flush=True)
    base = FlatCE(bcc_quaternary_ce())
    flat = _with_orbit(base, [(0, i % 5, i // 5, 0) for i in range(20)], 0)   # 4^20 decorations
    eng, occs = _loaded(flat, [(6, 6, 6)])
    ref = O.OracleSystem(base, (6, 6, 6)).corr(occs[0])
    assert np.abs(eng.correlations(0) - ref).max() <= 1e-12 * np.abs(ref).max()
    eng.close()

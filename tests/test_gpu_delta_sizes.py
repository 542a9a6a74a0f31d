"""Energy changes at the sizes where the call takes another route (read in
place up to 256 proposals, copied beyond, slices of 65,536) and with 1 to 4
sites, repeated and neighbouring sites among them, against the FP64 oracle.
The clusters are summed in FP64 over FP32 tables: FP32 rounding of at most a
few hundred table values, 1e-6 of the largest change plus 1e-6 eV."""
import numpy as np
import pytest

import oracle as O
from casmcode_clexmonte_amd.engine import Engine
from casmcode_clexmonte_amd.system import FlatCE, Supercell
from casmcode_clexmonte_amd.workloads import bcc_quaternary_ce, fcc_binary_ce, hcp_ternary_ce

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 3, 5, 256, 257, 65536, 65537])
@pytest.mark.parametrize("ce,m,chem", [(fcc_binary_ce, 1, True), (fcc_binary_ce, 2, False), (hcp_ternary_ce, 3, False),
                                       (bcc_quaternary_ce, 4, True)])
def test_delta_energy_sizes(n, ce, m, chem):
    print(f"[case] delta n={n} {ce.__name__} m={m} chem={chem}", flush=True)
    flat = FlatCE(ce())
    shapes = [Supercell(flat.ce.prim, d) for d in ((8, 7, 9), (7, 10, 8))]
    eng = Engine(flat)
    ids = [eng.add_supercell(sc, n_pair_phases=0) for sc in shapes]
    rng = np.random.default_rng(n + m)
    nocc = flat.n_occ_max
    occs = [rng.integers(0, nocc, sc.n_sites).astype(np.int8) for sc in shapes]
    w = rng.normal(0, 0.1, (2, flat.n_sublat, nocc))
    eng.load_chains(ids, occs, [600.0] * 2, [1, 2], chem=w)
    chain = rng.integers(0, 2, n)
    sites = rng.integers(0, 500, (n, m))
    if m > 1:
        sites[::3, 1] = sites[::3, 0]          # the same site twice
        sites[1::3, 1] = sites[1::3, 0] + 1    # neighbours
    new = rng.integers(0, nocc, (n, m))
    got = eng.delta_energy_batch(chain, sites, new, include_chem=chem)
    assert got.shape == (n,)
    osys = [O.OracleSystem(flat, sc.dims) for sc in shapes]
    ref, out = [], []
    for p in list(range(0, n, max(1, n // 40))) + [n - 1]:
        c = int(chain[p])
        d = osys[c].delta(occs[c], list(map(int, sites[p])), list(map(int, new[p])))
        if chem:
            cur = {}
            for s, v in zip(sites[p], new[p]):
                b = int(s) // shapes[c].n_cells
                d -= w[c, b, v] - w[c, b, cur.get(int(s), occs[c][s])]
                cur[int(s)] = v
        ref.append(d)
        out.append(got[p])
    assert np.abs(np.array(out) - np.array(ref)).max() <= 1e-6 * np.abs(ref).max() + 1e-6
    eng.close()

"""The N-fold kernel's routes: 64, 128 and 256 threads, a neighbour list
within one wavefront (FCC) and beyond it (BCC, 113 sites), lists with repeated
sites (small periodic cells), more than four groups of 64 rates per lane
(above 16,384 sites) and sampling by time.  Every block size gives the same
events bit for bit, and the energy and the counts are those of the state."""
import numpy as np
import pytest

import oracle as O
from casmcode_clexmonte_amd.engine import Engine
from casmcode_clexmonte_amd.system import FlatCE, Supercell
from casmcode_clexmonte_amd.workloads import bcc_quaternary_ce, fcc_binary_ce, hcp_ternary_ce

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("ce,dims,events", [
    (fcc_binary_ce, (12, 12, 12), 300), (fcc_binary_ce, (4, 5, 6), 200), (fcc_binary_ce, (26, 26, 25), 130),
    (hcp_ternary_ce, (6, 5, 6), 100), (bcc_quaternary_ce, (8, 9, 8), 70)])
@pytest.mark.parametrize("by_time", [False, True])
def test_nfold_block_sizes_agree(ce, dims, events, by_time):
    print(f"[case] nfold blocks {ce.__name__} {dims} by_time={by_time}", flush=True)
    flat = FlatCE(ce())
    sc = Supercell(flat.ce.prim, dims)
    rng = np.random.default_rng(2)
    occ = [rng.integers(0, flat.n_occ_max, sc.n_sites).astype(np.int8) for _ in range(2)]
    chem = rng.normal(0, 0.05, (2, flat.n_sublat * flat.n_occ_max))
    got = []
    for threads in (64, 128, 256, 0):
        eng = Engine(flat)
        sid = eng.add_supercell(sc, n_pair_phases=0)
        eng.load_chains([sid] * 2, occ, [700.0, 1400.0], [8, 9], chem=chem)
        eng.set_nfold_block_size(threads)
        if by_time:
            eng.nfold_run_time(10, 0.002, 100000)
            E, n = eng.read_samples()
            out = np.concatenate([E.ravel(), n.ravel()])
        else:
            out = eng.nfold_run_moments(events, 10)
        st = [eng.read_state(c) for c in range(2)]
        got.append((out, st))
        eng.close()
    osys = O.OracleSystem(flat, dims)
    for out, st in got:
        assert np.array_equal(out, got[0][0])
        for c in range(2):
            assert np.array_equal(st[c]["occ"], got[0][1][c]["occ"])
            assert st[c]["n_accept"] == got[0][1][c]["n_accept"] > 0
    for c in range(2):
        E = float(flat.eci @ osys.corr(got[0][1][c]["occ"]))
        tol = 1e-9 * abs(E) if flat.binary else 4e-6 * np.sqrt(got[0][1][c]["n_accept"]) + 1e-6
        assert abs(got[0][1][c]["E"] - E) <= tol
    if not by_time:
        assert got[0][1][0]["n_accept"] == events

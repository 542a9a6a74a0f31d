"""The N-fold block chosen by the number of chains: 256 + 64 threads while all
chains run at once, 128 + 64, and one wavefront for events and books (general
expansions not specialised: one or two always), which forms a group's sum in
one lane instead of four.  Every block gives the same
events and moments bit for bit (64 + 64 threads asked for as the comparison),
specialised or not, by events and by time, with lists of distinct and of
repeated neighbour sites.  A device has at least 200 and at most 320 compute
units here, which the chain counts allow for."""
import numpy as np
import pytest

from casmcode_clexmonte_amd.engine import Engine
from casmcode_clexmonte_amd.system import FlatCE, Supercell
from casmcode_clexmonte_amd.workloads import bcc_quaternary_ce, fcc_binary_ce, hcp_ternary_ce

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("ce,dims,chains,threads,events", [
    (fcc_binary_ce, (12, 12, 12), 200, 320, 20), (fcc_binary_ce, (8, 8, 8), 1000, 192, 20),
    (fcc_binary_ce, (8, 8, 8), 2600, 64, 20), (fcc_binary_ce, (4, 5, 6), 2600, 64, 40),
    (hcp_ternary_ce, (6, 5, 6), 200, 320, 20), (hcp_ternary_ce, (6, 5, 6), 700, 192, 10),
    (hcp_ternary_ce, (6, 5, 6), 2100, 64, 10), (bcc_quaternary_ce, (7, 7, 8), 2100, 64, 10)])
@pytest.mark.parametrize("specialize", [True, False])
@pytest.mark.parametrize("by_time", [False, True])
def test_nfold_block_by_chains(ce, dims, chains, threads, events, specialize, by_time):
    print(f"[case] nfold {ce.__name__} {dims} x {chains} by_time={by_time} specialize={specialize}", flush=True)
    flat = FlatCE(ce())
    sc = Supercell(flat.ce.prim, dims)
    rng = np.random.default_rng(6)
    occ = rng.integers(0, flat.n_occ_max, (chains, sc.n_sites)).astype(np.int8)
    chem = rng.normal(0, 0.05, (chains, flat.n_sublat * flat.n_occ_max))
    got = []
    for block in (0, 64):
        eng = Engine(flat)
        eng.set_specialization(specialize)
        sid = eng.add_supercell(sc, n_pair_phases=0)
        eng.load_chains([sid] * chains, list(occ), np.linspace(600.0, 1500.0, chains), np.arange(chains, dtype=np.uint64),
                        chem=chem)
        eng.set_nfold_block_size(block)
        if by_time:
            eng.nfold_run_time(3, 8.0 / sc.n_sites, 100000)
            E, n = eng.read_samples()
            out = np.concatenate([E.ravel(), n.ravel()])
        else:
            out = eng.nfold_run_moments(events, events // 2)
        info = eng.last_run_info()
        assert info["specialized"] == specialize
        want = threads if specialize or flat.binary else (64, 128)
        assert info["threads"] in ((128,) if block else np.atleast_1d(want))
        got.append((out, [eng.read_state(c) for c in range(0, chains, 97)]))
        eng.close()
    (a, sa), (b, sb) = got
    assert np.array_equal(a, b)
    for x, y in zip(sa, sb):
        assert np.array_equal(x["occ"], y["occ"])
        assert x["E"] == y["E"] and x["n_accept"] == y["n_accept"]
    assert sum(x["n_accept"] for x in sa) > 0

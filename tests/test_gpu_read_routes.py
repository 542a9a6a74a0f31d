"""Sample reads on both sides of their rules: rows side by side (four chains
and more up to 16,384 samples, fewer up to 512), two groups of rows (above
32 MiB), rows one by one, and a read after every short run while the samples
grow.  Every chain's sample at the end of a run is the state it was in then,
and a read repeats what an earlier one gave."""
import numpy as np
import pytest

from casmcode_clexmonte_amd.engine import Engine
from casmcode_clexmonte_amd.system import FlatCE, Supercell
from casmcode_clexmonte_amd.workloads import fcc_binary_ce, random_occupation

pytestmark = pytest.mark.gpu


def _engine(n_chains):
    flat = FlatCE(fcc_binary_ce())
    sc = Supercell(flat.ce.prim, (6, 6, 6))
    eng = Engine(flat)
    sid = eng.add_supercell(sc, n_pair_phases=0)
    eng.load_chains([sid] * n_chains, [random_occupation(sc.n_sites, 0.5, c) for c in range(n_chains)],
                    [900.0] * n_chains, list(range(n_chains)), chem=[[0.0, 0.05]] * n_chains)
    return eng


@pytest.mark.parametrize("n_chains,parts", [
    (100, [5000, 6000, 5000]), (4, [8000, 8384]), (4, [8000, 8385]), (3, [500, 12]), (3, [500, 13]), (2, [20000]),
    (7, [1, 2, 3, 50, 200, 1000, 3000])])
def test_rows_of_every_route(n_chains, parts):
    print(f"[case] sample rows, {n_chains} chains, {parts}", flush=True)
    eng = _engine(n_chains)
    seen, at = [], 0
    for n in parts:
        eng.run_passes("semigrand_canonical", n, 1)
        at += n
        seen.append((at, [eng.read_state(c) for c in range(n_chains)], eng.read_samples()))
    E, counts = seen[-1][2]
    assert E.shape == (n_chains, at) and counts.shape == (n_chains, at, 4)
    assert (counts.sum(2) == 216).all()
    for at, states, (E0, counts0) in seen:
        assert np.array_equal(E[:, :at], E0) and np.array_equal(counts[:, :at], counts0)
        for c, st in enumerate(states):
            assert E[c, at - 1] == st["E"]
            assert np.array_equal(counts[c, at - 1, :2], np.bincount(st["occ"], minlength=2))
    eng.close()

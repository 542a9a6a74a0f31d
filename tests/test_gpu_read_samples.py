"""Sample reads: several chains put side by side on the device, and single
long rows, both equal to the samples as the chains recorded them (the last
sample is the chain's state; reading in two parts gives the same rows)."""
import numpy as np
import pytest

from casmcode_clexmonte_amd.engine import Engine
from casmcode_clexmonte_amd.system import FlatCE, Supercell
from casmcode_clexmonte_amd.workloads import fcc_binary_ce, random_occupation

pytestmark = pytest.mark.gpu


def _run(n_chains, parts):
    flat = FlatCE(fcc_binary_ce())
    sc = Supercell(flat.ce.prim, (6, 6, 6))
    eng = Engine(flat)
    sid = eng.add_supercell(sc, n_pair_phases=0)
    occs = [random_occupation(sc.n_sites, 0.5, c) for c in range(n_chains)]
    eng.load_chains([sid] * n_chains, occs, [900.0] * n_chains, list(range(n_chains)), chem=[[0.0, 0.05]] * n_chains)
    for p in parts:
        eng.run_passes("semigrand_canonical", p, 1)
    E, cnt = eng.read_samples()
    last = [eng.read_state(c) for c in range(n_chains)]
    eng.close()
    return E, cnt, last


@pytest.mark.parametrize("n_chains", [1, 2, 5])
@pytest.mark.parametrize("n", [1, 3, 255, 256, 300])
def test_samples_of_several_chains(n_chains, n):
    print(f"[case] samples of {n_chains} chains x {n}", flush=True)
    E, cnt, last = _run(n_chains, [n])
    assert E.shape == (n_chains, n) and cnt.shape == (n_chains, n, 4)
    for c in range(n_chains):
        assert E[c, -1] == last[c]["E"]
        assert np.array_equal(cnt[c, -1, :2], np.bincount(last[c]["occ"], minlength=2))
        assert (cnt[c].sum(1) == 216).all()
        E1, cnt1, _ = _run(c + 1, [n]) if n_chains == 2 else (E, cnt, None)
        assert np.array_equal(E1[c], E[c]) and np.array_equal(cnt1[c], cnt[c])


def test_samples_long_rows():
    print("[case] samples, 800,000 per chain", flush=True)
    E, cnt, last = _run(2, [800000])   # more than half the group copy's bytes
    for c in range(2):
        assert E[c, -1] == last[c]["E"]
        assert np.array_equal(cnt[c, -1, :2], np.bincount(last[c]["occ"], minlength=2))
        assert (cnt[c].sum(1) == 216).all()

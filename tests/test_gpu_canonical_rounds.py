"""Canonical matchings: offsets drawn 64 at a time (more matchings per set, and
more sets, than that), set compositions counted per pass, and a class's
occupants kept side by side in LDS or, at the LDS limit, read through the
site addresses.  42x48x42 is such a supercell: its int8 image leaves no room
for them, its 2-bit image does, so the two runs take the two routes and must
agree bit for bit.  Final energies against the FP64 oracle's recompute."""
import numpy as np
import pytest

import oracle as O
from casmcode_clexmonte_amd.engine import Engine
from casmcode_clexmonte_amd.system import FlatCE, Supercell
from casmcode_clexmonte_amd.workloads import fcc_binary_ce, hcp_ternary_ce

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("ce,dims,rounds,passes", [
    (fcc_binary_ce, (42, 48, 42), 0, 2), (fcc_binary_ce, (42, 48, 42), 2, 2),
    (fcc_binary_ce, (10, 9, 7), 0, 4), (fcc_binary_ce, (10, 9, 7), 3, 4), (fcc_binary_ce, (12, 12, 12), 70, 2),
    (hcp_ternary_ce, (7, 5, 6), 0, 3), (hcp_ternary_ce, (8, 8, 6), 65, 1)])
def test_canonical_rounds_routes_agree(ce, dims, rounds, passes):
    print(f"[case] canonical rounds {ce.__name__} {dims} rounds={rounds}", flush=True)
    flat = FlatCE(ce())
    sc = Supercell(flat.ce.prim, dims)
    rng = np.random.default_rng(5)
    occ = [rng.integers(0, flat.n_occ_max, sc.n_sites).astype(np.int8) for _ in range(2)]
    res = []
    for packing in ("int8", "packed2"):
        eng = Engine(flat)
        sid = eng.add_supercell(sc, n_pair_phases=2)
        eng.load_chains([sid] * 2, occ, [500.0, 900.0], [1, 2])
        eng.set_image_packing(packing)
        eng.set_slabs(1)
        eng.run_passes("canonical", passes, 1, rounds)
        st = [eng.read_state(c) for c in range(2)]
        res.append((eng.read_samples(), st))
        eng.close()
    (Ea, na), sa = res[0]
    (Eb, nb), sb = res[1]
    assert np.array_equal(Ea, Eb) and np.array_equal(na, nb)
    osys = O.OracleSystem(flat, dims)
    for c in range(2):
        assert np.array_equal(sa[c]["occ"], sb[c]["occ"])
        assert sa[c]["n_accept"] == sb[c]["n_accept"] > 0 and sa[c]["n_attempt"] == sb[c]["n_attempt"]
        assert np.array_equal(np.bincount(sa[c]["occ"]), np.bincount(occ[c]))
        E = float(flat.eci @ osys.corr(sa[c]["occ"]))
        # binary: exact counts; general: FP32 changes summed in FP64
        assert abs(sa[c]["E"] - E) <= (1e-9 * abs(E) if flat.binary else 4e-6 * np.sqrt(sa[c]["n_accept"]) + 1e-6)

"""Full correlations by decoration counts: supercells below and above the
one-block form, cell ranges with a remainder, several shapes in one load,
against the FP64 oracle.  The counts are exact integers and the sum over
decorations is FP64: 1e-12 of the largest correlation."""
import numpy as np
import pytest

import oracle as O
from casmcode_clexmonte_amd.engine import Engine
from casmcode_clexmonte_amd.system import FlatCE, Supercell
from casmcode_clexmonte_amd.workloads import bcc_quaternary_ce, fcc_binary_ce, hcp_ternary_ce

pytestmark = pytest.mark.gpu

CES = {"fcc": fcc_binary_ce, "hcp": hcp_ternary_ce, "bcc": bcc_quaternary_ce}


@pytest.mark.parametrize("ce,shapes", [
    ("fcc", [(5, 5, 5)]), ("fcc", [(12, 12, 12)]), ("fcc", [(14, 14, 14)]), ("fcc", [(17, 18, 20)]),
    ("hcp", [(6, 6, 5), (13, 11, 12)]), ("hcp", [(16, 16, 10)]), ("bcc", [(7, 7, 7), (8, 9, 7)]),
    ("bcc", [(16, 17, 16)])])
def test_correlations_cell_ranges(ce, shapes):
    print(f"[case] correlations {ce} {shapes}", flush=True)
    flat = FlatCE(CES[ce]())
    eng = Engine(flat)
    scs = [Supercell(flat.ce.prim, d) for d in shapes]
    ids = [eng.add_supercell(sc, n_pair_phases=0) for sc in scs]
    rng = np.random.default_rng(3)
    occs = [rng.integers(0, flat.n_occ_max, sc.n_sites).astype(np.int8) for sc in scs]
    eng.load_chains(ids, occs, [900.0] * len(ids), list(range(len(ids))))
    for c, sc in enumerate(scs):
        ref = O.OracleSystem(flat, sc.dims).corr(occs[c])
        got = eng.correlations(c)
        assert np.abs(got - ref).max() <= 1e-12 * np.abs(ref).max()
        E = float(flat.eci @ ref)
        assert abs(eng.read_state(c)["E"] - E) <= 1e-9 * max(1.0, abs(E))
    eng.close()

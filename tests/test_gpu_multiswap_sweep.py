"""The fixed-composition sweep of a multiswap run is the canonical sweep: after
one pass with one multiswap attempt of at most two sites, the occupants differ
from those of one canonical pass with the same seeds at no more than two sites
(an accepted attempt changes its own sites; everything before it is the same
draws on the same image).  Sets of one and several wavefronts' sites, odd and
even cells, tables and slots, both image forms, both kernel builds."""
import numpy as np
import pytest

from casmcode_clexmonte_amd.engine import Engine
from casmcode_clexmonte_amd.system import FlatCE, Supercell, make_multiswaps
from casmcode_clexmonte_amd.workloads import bcc_quaternary_ce, fcc_binary_ce, hcp_ternary_ce

pytestmark = pytest.mark.gpu

CES = {"fcc": fcc_binary_ce, "hcp": hcp_ternary_ce, "bcc": bcc_quaternary_ce}


def _run(flat, dims, kind, rounds, packing, specialize, multiswaps):
    sc = Supercell(flat.ce.prim, dims)
    eng = Engine(flat)
    eng.set_specialization(specialize)
    eng.set_image_packing(packing)
    eng.set_slabs(1)
    eng.set_block_size(64)
    sid = eng.add_supercell(sc, n_pair_phases=2)
    rng = np.random.default_rng(3)
    occ = [rng.integers(0, flat.n_occ_max, sc.n_sites).astype(np.int8) for _ in range(3)]
    eng.load_chains([sid] * 3, occ, [500.0, 900.0, 1500.0], [5, 6, 7],
                    chem=np.zeros((3, flat.n_sublat, flat.n_occ_max)))
    if multiswaps:
        eng.set_multiswaps(multiswaps, per_pass=1)
    eng.run_passes(kind, 1, 1, canonical_rounds=rounds)
    out = [eng.read_state(c)["occ"] for c in range(3)]
    eng.close()
    return occ, out


@pytest.mark.parametrize("packing,specialize", [("int8", True), ("packed2", True), ("int8", False)])
@pytest.mark.parametrize("rounds", [0, 4])
@pytest.mark.parametrize("ce,dims", [
    ("fcc", (8, 8, 8)), ("fcc", (7, 5, 9)), ("fcc", (24, 24, 24)), ("bcc", (10, 10, 7)), ("hcp", (9, 8, 7))])
def test_sweep_is_the_canonical_one(ce, dims, rounds, packing, specialize):
    print(f"[case] multiswap sweep {ce} {dims} rounds {rounds} {packing} {specialize}", flush=True)
    flat = FlatCE(CES[ce]())
    start, a = _run(flat, dims, "canonical", rounds, packing, specialize, None)
    _, b = _run(flat, dims, "semigrand_canonical", rounds, packing, specialize, make_multiswaps(flat, 2))
    for s, x, y in zip(start, a, b):
        assert (s != x).sum() > 2
        assert (x != y).sum() <= 2

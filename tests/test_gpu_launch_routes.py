"""Which kernel a launch takes at the lines of its rules: spread fields for sets
of at most 8 sites (specialised, one wavefront per chain, tables, unpacked), and
a set's occupants in LDS during canonical matchings where the image leaves room.
42 x 48 x 42 is a supercell whose int8 image does not."""
import numpy as np
import pytest

from casmcode_clexmonte_amd.engine import Engine
from casmcode_clexmonte_amd.system import FlatCE, Supercell, color_classes
from casmcode_clexmonte_amd.workloads import bcc_quaternary_ce, fcc_binary_ce, hcp_ternary_ce

pytestmark = pytest.mark.gpu

CES = {"fcc": fcc_binary_ce, "hcp": hcp_ternary_ce, "bcc": bcc_quaternary_ce}


def _run(ce, dims, kind, packing="auto", specialize=True, block=0):
    flat = FlatCE(CES[ce]())
    sc = Supercell(flat.ce.prim, dims)
    eng = Engine(flat)
    eng.set_specialization(specialize)
    eng.set_image_packing(packing)
    eng.set_slabs(1)
    sid = eng.add_supercell(sc, n_pair_phases=0)
    rng = np.random.default_rng(1)
    eng.load_chains([sid] * 2, [rng.integers(0, flat.n_occ_max, sc.n_sites).astype(np.int8) for _ in range(2)],
                    [900.0] * 2, [1, 2])
    eng.set_block_size(block)
    eng.run_passes(kind, 1, 1, 1)
    out = eng.last_run_routes(), eng.last_run_info()
    eng.close()
    return out, max(len(c) for c in color_classes(flat, sc))


@pytest.mark.parametrize("kind", ["canonical", "semigrand_canonical"])
@pytest.mark.parametrize("ce,dims,sites", [
    ("hcp", (8, 7, 7), 2), ("hcp", (11, 9, 7), 3), ("hcp", (9, 10, 7), 6), ("bcc", (10, 10, 7), 4), ("bcc", (8, 8, 10), 8),
    ("hcp", (7, 9, 9), 9), ("bcc", (10, 10, 9), 12), ("fcc", (7, 5, 9), 0)])
def test_spread_fields_up_to_eight_sites(ce, dims, sites, kind):
    print(f"[case] spread route {ce} {dims} {kind}", flush=True)
    (routes, info), n_max = _run(ce, dims, kind)
    assert info["specialized"] and info["threads"] == 64
    assert sites in (0, n_max)
    assert routes["spread"] == (ce != "fcc" and n_max <= 8)
    for kw in ({"specialize": False}, {"packing": "packed2"}, {"block": 128}):
        assert not _run(ce, dims, kind, **kw)[0][0]["spread"]


@pytest.mark.parametrize("packing,kept", [("int8", False), ("packed2", True)])
def test_occupants_of_a_set_in_lds_where_they_fit(packing, kept):
    print(f"[case] class occupants {packing}", flush=True)
    (routes, _), _ = _run("fcc", (42, 48, 42), "canonical", packing)
    assert routes["class_occ"] == kept
    (routes, _), _ = _run("fcc", (12, 12, 12), "canonical", packing)
    assert routes["class_occ"]
    (routes, _), _ = _run("fcc", (12, 12, 12), "semigrand_canonical", packing)
    assert not routes["class_occ"]

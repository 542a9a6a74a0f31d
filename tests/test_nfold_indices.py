"""The N-fold kernel's LDS layout and index arithmetic, compiled for the host
(tests/cpp/nfold_index_check): regions that do not overlap, the rates' places
and the groups' sums, the quick divisions, the periodic copies and neighbours
of every site, in the image's bounds, for the shapes that the GPU tests run,
supercells smaller than their halo and the largest the LDS holds; and shapes
made up at the limits of the byte offsets (halo 26) and of the divisions
(one long axis).  None of it depends on the number of threads."""
import os
import subprocess

import numpy as np
import pytest

from casmcode_clexmonte_amd.system import FlatCE, interaction_offsets
from casmcode_clexmonte_amd.workloads import bcc_quaternary_ce, fcc_binary_ce, fcc_ordering_ce, hcp_ternary_ce

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CHECK = os.path.join(ROOT, "tests", "cpp", "nfold_index_check")
MAX_LDS = 160 * 1024


def _lists(flat):
    offs = interaction_offsets(flat)
    out = []
    for b in range(flat.n_sublat):
        rest = sorted({tuple(int(v) for v in o) for o in offs.get(b, [])} - {(b, 0, 0, 0)})
        out.append([(b, 0, 0, 0)] + rest)
    return out


def _shape(lists, dims, pitch=0, halo=None):
    h = max(abs(v) for l in lists for o in l for v in o[1:]) if halo is None else halo
    lines = [f"{len(lists)} {dims[0]} {dims[1]} {dims[2]} {h} {pitch}"]
    for l in lists:
        lines.append(str(len(l)) + " " + " ".join(f"{b} {i} {j} {k}" for b, i, j, k in l))
    return "\n".join(lines)


def _run(shapes):
    r = subprocess.run([CHECK], input="\n".join(shapes) + "\n", capture_output=True, text=True, check=True)
    rows = [l.split() for l in r.stdout.splitlines()]
    assert len(rows) == len(shapes)
    return [(int(x[1]), int(x[3])) for x in rows]


@pytest.mark.skipif(not os.path.exists(CHECK), reason="tests/cpp/nfold_index_check not built (run build())")
@pytest.mark.parametrize("ce,dims", [
    (fcc_binary_ce, [(4, 5, 6), (8, 8, 8), (12, 12, 12), (24, 24, 24), (26, 26, 25), (2, 1, 3), (1, 1, 1)]),
    (fcc_ordering_ce, [(4, 4, 4), (16, 16, 16)]),
    (hcp_ternary_ce, [(6, 5, 6), (4, 4, 3), (12, 12, 8), (2, 2, 1), (20, 20, 16)]),
    (bcc_quaternary_ce, [(8, 9, 8), (7, 7, 8), (2, 3, 2), (1, 5, 9)])])
def test_indices_of_the_tested_shapes(ce, dims):
    lists = _lists(FlatCE(ce()))
    for lds, errors in _run([_shape(lists, d, p) for d in dims for p in (0, 3)]):
        assert lds <= MAX_LDS and errors == 0


@pytest.mark.skipif(not os.path.exists(CHECK), reason="tests/cpp/nfold_index_check not built (run build())")
def test_indices_at_the_limits():
    rng = np.random.default_rng(1)
    far = [(0, 0, 0, 0)] + [tuple([0] + list(rng.integers(-26, 27, 3))) for _ in range(200)] + [(0, 26, -26, 26)]
    # (the largest halo leaves room for an image of one cell per axis and its rates only)
    assert _run([_shape([far], (1, 1, 1), halo=26)])[0][1] == 0
    pair = [(0, 0, 0, 0), (0, 1, 0, 0), (0, -1, 0, 0)]
    long = [(2700, 1, 1), (1, 2700, 1), (1, 1, 2700), (3, 400, 2)]
    for lds, errors in _run([_shape([pair], d, halo=1) for d in long]):
        assert lds <= MAX_LDS and errors == 0
    # cells of 2^14 and more (one sublattice, no halo), an axis longer than any index
    alone = [(0, 0, 0, 0)]
    for lds, errors in _run([_shape([alone], d, halo=0) for d in [(20000, 1, 1), (1, 20000, 1), (2, 2, 7900), (17, 1000, 1)]]):
        assert lds <= MAX_LDS and errors == 0

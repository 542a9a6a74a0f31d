"""Pair phases of the grouped proposals with more pairs than random streams:
every pair of a phase is accepted or rejected with a random word of its own.

Occupants uniform within every independent set leave the grouped proposals
nothing to swap, so the first pass is its pair phases alone, and each pair's
word is known: Philox at (pair's place in the phase, counter of its stream,
chain).  The moves are replayed in FP64 with the oracle's energy changes and
must come out the same, site by site.  FP32 fields and exponentials are good
to 1e-5 of the acceptance probability; no word of these seeds lies that close
to its threshold.  Blocks of 64 and 128 threads have fewer streams than the
225 pairs of the phase, 256 has more."""
import numpy as np
import pytest

import oracle as O
from casmcode_clexmonte_amd.engine import Engine, pair_phases
from casmcode_clexmonte_amd.system import KB, BasisSet, ClusterExpansion, FlatCE, Prim, Supercell, color_classes
from casmcode_clexmonte_amd.workloads import random_mlp_params

pytestmark = pytest.mark.gpu

DIMS = (12, 12, 12)


def _flat():
    prim = Prim(np.eye(3).tolist(), [[0, 0, 0]], [["A", "B"]])
    bs = BasisSet(prim, {2: 1.01}, "chebychev")   # simple cubic, nearest-neighbour pairs
    eci = np.zeros(bs.n_functions)
    eci[-1] = 0.03
    return FlatCE(ClusterExpansion(bs, eci))


def _replay(flat, sc, occ, T, seed, chain, block, rounds):
    """Final occupation and accepted swaps of one pass of pair phases."""
    osys = O.OracleSystem(flat, sc.dims)
    key = [seed & 0xFFFFFFFF, seed >> 32]
    phase = pair_phases(flat, sc, 1, 0)[0]
    streams = block // 64
    groups = [(len(c) + 63) // 64 for c in color_classes(flat, sc)]
    draw = [sum((g - s + streams - 1) // streams for g in groups) * 64 * ((rounds + 15) // 16) for s in range(streams)]
    n_rounds = -(-sc.n_sites // (4 * len(phase)))
    occ, accepted, margin = occ.copy(), 0, 1.0
    for rd in range(n_rounds):
        for i, (s, t) in enumerate(phase.tolist()):
            if occ[s] == occ[t]:
                continue
            d = draw[(i % block) // 64] + rd
            u = O.philox4x32_10([i, d, 0x80000000, chain], key)[0] / 2.0 ** 32
            p = np.exp(-osys.delta(occ, [s, t], [int(occ[t]), int(occ[s])]) / (KB * T))
            margin = min(margin, abs(u - p))
            if u < p:
                occ[s], occ[t] = occ[t], occ[s]
                accepted += 1
    return occ, accepted, margin


@pytest.mark.parametrize("proposal", ["grouped_uniform", "learned", "informed"])
@pytest.mark.parametrize("block", [64, 128, 256])
def test_every_pair_has_its_own_word(block, proposal):
    print(f"[case] pair words {proposal} block={block}", flush=True)
    flat = _flat()
    sc = Supercell(flat.ce.prim, DIMS)
    occ = np.zeros(sc.n_sites, dtype=np.int8)
    occ[color_classes(flat, sc)[1]] = 1
    T, seeds, rounds = [2000.0, 3500.0], [11, (5 << 32) + 12], 16
    eng = Engine(flat)
    sid = eng.add_supercell(sc, n_pair_phases=1, seed=0)
    eng.load_chains([sid] * 2, [occ, occ], T, seeds)
    eng.mlp_set_params(random_mlp_params(2, eng.mlp_info()[0]))
    eng.set_proposal(proposal, rounds_per_group=rounds)
    eng.set_block_size(block)
    eng.run_passes("canonical", 1, 1)
    for c in range(2):
        st = eng.read_state(c)
        ref, accepted, margin = _replay(flat, sc, occ, T[c], seeds[c], c, block, rounds)
        assert margin > 1e-5 and accepted > 20
        assert st["n_accept"] == accepted
        assert np.array_equal(st["occ"], ref)
    eng.close()

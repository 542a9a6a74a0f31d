"""Grouped proposals with one and with two wavefronts per random stream: chains
that share the device one per compute unit take twice the threads, more chains
do not.  A chain's moves depend on its own number and seed only, so the first
100 of 300 chains (256 compute units) make the moves that 100 chains alone
make, bit for bit: sets with one group of 64 sites, with several groups per
stream (blocks of 64 threads), pair phases and semi-grand canonical flips."""
import numpy as np
import pytest
import torch

from casmcode_clexmonte_amd.engine import Engine
from casmcode_clexmonte_amd.system import FlatCE, Supercell
from casmcode_clexmonte_amd.workloads import fcc_ordering_ce, random_mlp_params

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dims,block", [((12, 12, 12), 0), ((16, 16, 16), 64), ((15, 12, 14), 128)])
@pytest.mark.parametrize("kind", ["canonical", "semigrand_canonical"])
@pytest.mark.parametrize("proposal", ["learned", "informed", "grouped_uniform"])
def test_chain_moves_do_not_depend_on_the_number_of_chains(dims, block, kind, proposal):
    print(f"[case] grouped {proposal} {kind} {dims} block={block}", flush=True)
    few, many = 100, 300
    assert few <= torch.cuda.get_device_properties(0).multi_processor_count < many
    flat = FlatCE(fcc_ordering_ce())
    sc = Supercell(flat.ce.prim, dims)
    rng = np.random.default_rng(4)
    occ = rng.integers(0, 2, (many, sc.n_sites)).astype(np.int8)
    chem = np.zeros((many, flat.n_sublat, flat.n_occ_max))
    chem[:, :, 1] = 0.05
    got = []
    for n in (few, many):
        eng = Engine(flat)
        sid = eng.add_supercell(sc, n_pair_phases=3, seed=2)
        eng.load_chains([sid] * n, list(occ[:n]), np.linspace(150.0, 700.0, many)[:n], np.arange(n, dtype=np.uint64),
                        chem=chem[:n])
        eng.mlp_set_params(random_mlp_params(5, eng.mlp_info()[0]))
        eng.set_proposal(proposal, rounds_per_group=16)
        eng.set_block_size(block)
        eng.run_passes(kind, 3, 1)
        E, counts = eng.read_samples()
        got.append((E[:few], counts[:few], [eng.read_state(c) for c in range(0, few, 9)]))
        eng.close()
    (Ea, na, sa), (Eb, nb, sb) = got
    assert np.array_equal(Ea, Eb) and np.array_equal(na, nb)
    for x, y in zip(sa, sb):
        assert np.array_equal(x["occ"], y["occ"])
        assert x["E"] == y["E"] and x["n_accept"] == y["n_accept"] and x["n_attempt"] == y["n_attempt"]
    assert sum(x["n_accept"] for x in sa) > 0

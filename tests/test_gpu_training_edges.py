"""Training at its edges.  Gradients with values that are not finite: unused
inputs keep a zero gradient, and the rows that fill up a tile of 16 samples add
nothing.  Collected samples replayed one by one (site choice by the same Philox
words, features by the environment, labels by the oracle's flip energies, FP32
to 2e-5), with the occupation in LDS and, above 49,152 sites, in global memory,
at batch sizes around a block's 222 samples and on the smallest of cells."""
import numpy as np
import pytest

import oracle as O
from casmcode_clexmonte_amd.engine import Engine
from casmcode_clexmonte_amd.system import KB, FlatCE, Supercell
from casmcode_clexmonte_amd.workloads import fcc_binary_ce, random_mlp_params, random_occupation

pytestmark = pytest.mark.gpu


def test_unused_inputs_keep_a_zero_gradient():
    print("[case] gradients, a sample that is not finite", flush=True)
    eng = Engine(FlatCE(fcc_binary_ce()))
    n_env = eng.mlp_info()[0]
    rng = np.random.default_rng(0)
    eng.mlp_set_params(random_mlp_params(1, n_env, scale=0.8))
    X = rng.choice(np.array([-1, 1], np.int8), (40, 48))
    y = rng.random(40).astype(np.float32)
    y[7] = np.nan
    t = np.ones(40, np.float32)
    t[21] = np.inf
    g, _ = eng.mlp_gradients(X, y, t)
    W1 = g[:64 * 48].reshape(64, 48)
    assert np.all(W1[:, n_env:] == 0) and not np.isfinite(W1[:, :n_env]).all()
    eng.close()


def test_rows_past_the_batch_add_nothing():
    print("[case] gradients, an infinite bias", flush=True)
    eng = Engine(FlatCE(fcc_binary_ce()))
    n_env = eng.mlp_info()[0]
    p = np.zeros(3201)
    p[64 * 48 + 3] = np.inf          # unit 3 is infinite for every sample
    p[64 * 48 + 64 + 3] = 1.0        # and drives the output
    eng.mlp_set_params(p)
    g, _ = eng.mlp_gradients(np.ones((1, 48), np.int8), np.array([0.25], np.float32), None)
    # p = 1: dl = 0.75, times the infinite unit
    assert g[64 * 48 + 64 + 3] == np.inf and g[64 * 48 + 3] == np.float32(0.75) and g[3200] == np.float32(0.75)
    eng.close()


@pytest.mark.parametrize("dims,n", [((6, 5, 7), 1), ((6, 5, 7), 222), ((6, 5, 7), 223), ((6, 5, 7), 445), ((3, 4, 3), 60),
                                    ((36, 36, 37), 30), ((37, 37, 37), 30), ((37, 37, 37), 223)])
def test_collected_samples_replayed(dims, n):
    print(f"[case] collect {dims} n={n}", flush=True)
    flat = FlatCE(fcc_binary_ce())
    sc = Supercell(flat.ce.prim, dims)
    eng = Engine(flat)
    sid = eng.add_supercell(sc, n_pair_phases=0)
    T, mu, seeds = [700.0, 1300.0], 0.02, [5, (3 << 32) + 6]
    occs = [random_occupation(sc.n_sites, 0.4, 3), random_occupation(sc.n_sites, 0.5, 4)]
    eng.load_chains([sid] * 2, occs, T, seeds, chem=[[0.0, mu]] * 2)
    X, y, t = eng.mlp_collect(n, seed=9, include_chem=True)
    n_env, _, env = eng.mlp_info()
    osys = O.OracleSystem(flat, dims)
    L1, L2, _ = dims
    for c in range(2):
        beta, key = 1.0 / (KB * T[c]), [seeds[c] & 0xFFFFFFFF, seeds[c] >> 32]
        prob = {}

        def label(l):
            if l not in prob:
                dE = osys.delta(occs[c], [l], [1 - int(occs[c][l])]) - (mu if occs[c][l] == 0 else -mu)
                prob[l] = 1.0 / (1.0 + np.exp(beta * dE))
            return prob[l]

        for s in range(n):
            words = O.philox4x32_10([s, 9, 0xC011EC7, c], key) + O.philox4x32_10([s, 9, 0xC011EC8, c], key)
            cand = [w % sc.n_sites for w in words[:8 if s & 1 else 1]]
            row = c * n + s
            best = max(label(l) for l in cand)
            assert abs(y[row] - best) <= 2e-5 and abs(t[row] - 0.1 * beta) <= 1e-6 * beta
            # the site: any candidate within the labels' rounding of the best
            feats = []
            for l in cand:
                if label(l) < best - 4e-5:
                    continue
                i, j, k = l % L1, (l // L1) % L2, l // (L1 * L2)
                feats.append([1 if occs[c][sc.linear_index(b, i + di, j + dj, k + dk)] == occs[c][l] else -1
                              for b, di, dj, dk in env[0, :n_env].tolist()])
            assert list(X[row, :n_env]) in feats and not X[row, n_env:].any()
    eng.close()

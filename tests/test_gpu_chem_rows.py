"""Chemical potential and densities from the row-order passes at their edges,
against the oracle: H counts with every remainder modulo four, lanes per site
1..16, workgroups of 256, 512 and 1024 lanes, both rules, packets whose nodes
leave the tables' [1, 6) A, and nonzero correction terms.

Bar as elsewhere: 1e-10 of max(|gamma|, 1); densities 1e-10."""
import numpy as np
import pytest

import a2c_amd as A
import oracle as O
from helpers import specimen

pytestmark = pytest.mark.gpu

COE = np.array([0.3, 0.0, 0.2, -0.1]), np.array([0.5, 0.07, -0.03, 0.02])


@pytest.mark.parametrize("cells,npd,nh,lanes,quad,sigma", [
    (3, 1, 1, 1, "r12", (0.08, 0.15)),
    (3, 7, 6, 16, "gh3", (0.08, 0.15)),
    (5, 300, 65, 2, "r12", (0.08, 0.15)),
    (5, 0, 259, 4, "r12", (0.08, 0.15)),
    (4, 100, 90, 2, "r12", (0.30, 0.50)),
    (4, 100, 91, 8, "gh3", (0.20, 0.35)),
    (13, 8788, 8788, 1, "r12", (0.08, 0.15)),
    (13, 8788, 8788, 8, "gh3", (0.08, 0.15)),
    (13, 8788, 8786, 16, "r12", (0.08, 0.15)),
])
def test_edges(cells, npd, nh, lanes, quad, sigma):
    seed = npd + nh
    X, x, box, per, p, h = specimen(cells, seed=seed, disp=0.03, sigma=sigma, x=(0.01, 0.6), periodic=False)
    rng = np.random.default_rng(seed)
    ip, ih = np.sort(rng.permutation(p)[:npd]), np.sort(rng.permutation(h)[:nh])
    X = X.reshape(-1, 4)
    X, x = np.concatenate([X[ip], X[p + ih]]).reshape(-1), x[ih]
    orc = O.Oracle(npd, nh, box, per, T=400.0, threads=8, quad=quad)
    orc.build_neighbors(X)
    full = np.zeros(nh, np.int32)
    full[::13] = 1
    go, fo = orc.chem_potential(X, x, *COE, 1e9, np.full(nh, 3.0), full.copy())
    ro = orc.density(X, x)
    try:
        A.tune_set({"max_sites": [2**31 - 1], "lanes_mixed": [lanes], "lanes_fp64": [lanes]})
        with A.FreeEntropy(npd, nh, box, per, T=400.0, quad=quad) as fe:
            fe.set_occupancy(x)
            fe.findNeighbors(X)
            g, f = fe.calculateChemicalPotential(X, *COE, 1e9, np.full(nh, 3.0), full.copy())
            assert np.array_equal(f, fo)
            assert np.max(np.abs(g - go) / np.maximum(np.abs(go), 1.0)) <= 1e-10
            assert np.max(np.abs(fe.density(X) - ro)) <= 1e-10 * np.abs(ro).max()
    finally:
        A.tune_set(None)

"""One pair alone in the mixed evaluation against 50 digits, at distances that put
nodes on both sides of 1.8 A (below it Pd-Pd pairs are taken node by node from the
Hermite tables), of the joints, and past 6 A.

The bar: 64 2^-24 = 3.8e-6 of the sum of the terms' magnitudes.  A function costs
about four FP32 roundings of itself and an argument two or three of r, times r
|y'| / |y| of up to 10 at these distances."""
import numpy as np
import pytest

import a2c_amd as A
from eam_exact import D
from test_gpu_pair_exact import KINDS, OCC, SIGMA, T, objective

pytestmark = pytest.mark.gpu

DISTANCES = [1.45, 1.7, 1.8, 1.9, 2.1, 2.75, 4.0, 5.04, 5.3, 5.9]
BAR = 64 * 2.0 ** -24


@pytest.mark.parametrize("rule", ["r12", "gh3"])
@pytest.mark.parametrize("kind", list(KINDS))
def test_one_pair(kind, rule):
    direction = np.array([0.48, -0.6, 0.64])
    sp = KINDS[kind]
    npd = 2 - sum(sp)
    with A.FreeEntropy(npd, 2 - npd, (0, 0, 0), (0, 0, 0), T=T, rc=6.2, quad=rule, precision="mixed") as fe:
        fe.set_occupancy(np.array([OCC[k] for k in (0, 1) if sp[k]]))
        for dist in DISTANCES:
            X = np.concatenate([dist * direction, [SIGMA[0]], [0.0, 0.0, 0.0, SIGMA[1]]])
            fe.findNeighbors(X)
            f, G = fe.formFunctionAndGradient(X)
            for c in range(8):
                want, mag, dmag = objective(kind, rule, X, np.eye(8)[c])
                if c == 0:
                    assert abs(float(D(f) - want.v)) <= BAR * mag, (dist, f, float(want.v), mag)
                assert abs(float(D(G[c]) - want.d)) <= BAR * dmag, (dist, c, G[c], float(want.d), dmag)

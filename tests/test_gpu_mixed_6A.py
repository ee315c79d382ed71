"""A mixed evaluation with nodes at the end of the tables: a node whose |r|^2 rounds to
36 A^2 or just past it is beyond 6 A, and is evaluated by the exponential tail
whatever its rounded radius is.

One pair along x with the outermost node from 3e-6 A below 6 A to 3e-6 A above it, in
steps of a quarter of an FP32 unit there; against the FP64 evaluation to 3.8e-6
(64 2^-24) of the largest term, and finite (a2c_fe_eval refuses other objectives)."""
import numpy as np
import pytest

import a2c_amd as A

pytestmark = pytest.mark.gpu

SIGMA = (0.11, 0.08)
OUT = {"r12": np.sqrt(6.0) * SIGMA[0], "gh3": np.sqrt(3.0 * (SIGMA[0] ** 2 + SIGMA[1] ** 2))}


@pytest.mark.parametrize("rule", ["r12", "gh3"])
@pytest.mark.parametrize("n_pd", [2, 1, 0])
def test_nodes_around_6A(n_pd, rule):
    args = (n_pd, 2 - n_pd, (0, 0, 0), (0, 0, 0))
    kw = dict(T=400.0, rc=6.2, quad=rule)
    with A.FreeEntropy(*args, precision="mixed", **kw) as m, A.FreeEntropy(*args, precision="fp64", **kw) as d:
        for fe in (m, d):
            fe.set_occupancy(np.full(2 - n_pd, 0.4))
        for step in np.arange(-3e-6, 3e-6, 1.2e-7):
            X = np.array([6.0 - OUT[rule] + step, 0.0, 0.0, SIGMA[0], 0.0, 0.0, 0.0, SIGMA[1]])
            out = []
            for fe in (m, d):
                fe.findNeighbors(X)
                out.append(fe.formFunctionAndGradient(X))
            (f, G), (f0, G0) = out
            assert abs(f - f0) <= 64 * 2.0 ** -24 * abs(f0), step
            assert np.max(np.abs(G - G0)) <= 64 * 2.0 ** -24 * np.max(np.abs(G0)), step

"""Receive passes around the size where they change from four lanes per row to
one (32,768 sites) and in one batch that holds both kinds and an empty
lattice: against the full-list densities' objective of the oracle, and bit for
bit the same alone and in a batch.

Bars as elsewhere: FP64 objective 1e-10, gradient 1e-8; mixed 1e-7 and 1e-5."""
import numpy as np
import pytest

import a2c_amd as A
import oracle as O
from helpers import specimen

pytestmark = pytest.mark.gpu

SIZES = ((16383, 16385), (16384, 16385), (16500, 17001), (3, 2), (130, 127), (0, 0))


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
def test_sizes_alone_and_together(precision):
    X, x, box, per, p, h = specimen(17, seed=4, disp=0.03, sigma=(0.08, 0.15), x=(0.01, 0.6), periodic=False)
    X = X.reshape(-1, 4)
    lat = [(np.concatenate([X[:a], X[p:p + b]]).reshape(-1), x[:b], a, b) for a, b in SIZES]
    with A.Batch(precision=precision, max_lattices=len(lat)) as batch:
        slots = [batch.add(q, w, a, b, box, per, T=400.0) for q, w, a, b in lat]
        f = batch.eval(slots, precision)
        G = [batch.get_state(s)[1] for s in slots]
    for k, (q, w, a, b) in enumerate(lat):
        if a + b == 0:
            assert f[k] == 0.0
            continue
        with A.FreeEntropy(a, b, box, per, T=400.0, precision=precision) as fe:
            fe.set_occupancy(w)
            fe.findNeighbors(q)
            f1, G1 = fe.eval(q)
        assert f1 == f[k] and np.array_equal(G1, G[k])
        orc = O.Oracle(a, b, box, per, T=400.0, threads=8)
        orc.build_neighbors(q)
        fo, Go = orc.eval(q, w)
        if precision == "fp64":
            assert abs(f1 - fo) <= 1e-10 * abs(fo)
            assert np.max(np.abs(G1 - Go)) <= 1e-8 * np.abs(Go).max()
        else:
            assert abs(f1 - fo) <= 1e-7 * abs(fo)
            assert np.linalg.norm(G1 - Go) <= 1e-5 * np.linalg.norm(Go)

"""A captured evaluation is replayed only for a launch of the same kernels.

Lattices of 64 + 64 and 64 + 64 sites and of 0 and 128 + 128 have the same site
blocks and owner units, but an empty lattice keeps the row-order copies (and the
clearing of its count of finished blocks) in a launch of their own.  With
graphs on, the second pair evaluated after the first must not be the first one's
replay: the empty lattice's objective is 0, not what its slot held before."""
import numpy as np
import pytest

import a2c_amd as A
from helpers import specimen

pytestmark = pytest.mark.gpu


def cut(n, seed):
    """n Pd and n H sites of a free specimen"""
    X, x, box, per, p, h = specimen(4, seed=seed, disp=0.02, sigma=(0.09, 0.12), x=(0.05, 0.6), periodic=False)
    X = X.reshape(-1, 4)
    return dict(X=np.concatenate([X[:n], X[p:p + n]]).reshape(-1), x=x[:n], n_pd=n, n_h=n, box=box, periodic=per, T=400.0)


@pytest.mark.parametrize("precision", ["mixed", "fp64"])
def test_an_empty_lattice_in_a_captured_launch(precision):
    small, large, empty = [cut(64, 1), cut(64, 2)], cut(128, 3), cut(0, 4)
    with A.Batch(precision=precision, graphs=False) as b:
        f_large = b.eval([b.add(**large)], precision=precision)[0]
    with A.Batch(precision=precision, graphs=True, max_lattices=3) as b:
        slots = [b.add(**s) for s in small]
        big = b.add(**large)
        for _ in range(4):
            f = b.eval(slots, precision=precision)
            assert np.all(f != 0.0)
        assert b.graph_stats()["captures"] == 1
        b.remove(slots[0])
        assert b.add(**empty) == slots[0]
        for _ in range(4):
            f = b.eval([slots[0], big], precision=precision)
            assert f[0] == 0.0 and f[1] == f_large

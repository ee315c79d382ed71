"""The cell walk at the edges of its filter and its lane split, against the
oracle's sets, bit for bit: grids of 1, 2, 3 and more cells per axis, open
and periodic; rows from 0 to about 250 neighbors; site counts around the
rows of a workgroup; sites outside the periodic box and far from the origin;
pairs exactly at the cutoff.  Both the first build and the second, whose skin
lists come from the same walk."""
import numpy as np
import pytest

import a2c_amd as A
import oracle as O

pytestmark = pytest.mark.gpu


def cloud(shape, spacing, jitter, seed, offset=0.0):
    rng = np.random.default_rng(seed)
    q = np.stack(np.meshgrid(*(np.arange(n) for n in shape), indexing="ij"), -1).reshape(-1, 3) * spacing
    q = q + rng.uniform(-jitter, jitter, q.shape) + offset
    return q[rng.permutation(len(q))], rng


@pytest.mark.parametrize("shape,spacing,jitter,npd,periodic,offset,images", [
    ((1, 1, 1), 1.0, 0.0, 1, (0, 0, 0), 0.0, 0),
    ((5, 13, 1), 1.4, 0.05, 33, (0, 0, 0), 3.0, 0),        # one cell across an axis, 65 sites
    ((8, 8, 8), 1.42, 0.05, 250, (1, 1, 1), 0.0, 2),       # one periodic cell, rows near 225
    ((9, 9, 9), 1.42, 0.02, 31, (0, 0, 0), -1e5, 0),       # two cells per axis
    ((10, 9, 11), 1.9, 0.2, 500, (1, 0, 1), 0.0, 3),       # sites in other images of the box
    ((2, 3, 150), 2.5, 0.3, 449, (0, 0, 0), 1e4, 0),       # a column of cells
    ((7, 7, 7), 2.675, 0.0, 100, (0, 0, 0), 0.0, 0),       # pairs at exactly rc = 5.35
    ((9, 9, 9), 2.675, 0.0, 365, (1, 1, 1), 0.0, 1),
    ((20, 20, 20), 1.9, 0.1, 4000, (1, 1, 1), 0.0, 0),
])
def test_sets(shape, spacing, jitter, npd, periodic, offset, images):
    q, rng = cloud(shape, spacing, jitter, 5, offset)
    box = np.array(shape) * spacing
    if images:
        q = q + rng.integers(-images, images + 1, q.shape) * box * np.array(periodic)
    N = len(q)
    X = np.concatenate([q, np.full((N, 1), 0.1)], 1).reshape(-1)
    orc = O.Oracle(npd, N - npd, box, periodic, threads=8)
    mx = orc.build_neighbors(X)
    with A.FreeEntropy(npd, N - npd, box, periodic) as fe:
        fe.set_occupancy(np.full(N - npd, 0.3))
        for _ in range(2):
            st = fe.findNeighbors(X)
            assert st["max_neib"] == mx
            for w in ("PdPd", "PdH", "HPd", "HH", "HH1"):
                go, gi = fe.neighbors(w)
                oo, oi = orc.neighbors(w)
                assert np.array_equal(go, oo) and np.array_equal(gi, oi), w
            assert np.array_equal(fe.pdpdnum(), orc.pdpdnum())

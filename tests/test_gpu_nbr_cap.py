"""Rows at the neighbor cap: 255, 256 and 257 neighbors within the cutoff of every
site, as one species or split over both.  Up to 256 the lists are the oracle's, bit
for bit, from the cell walk and from the skin lists; 257 are refused."""
import numpy as np
import pytest

import a2c_amd as A
import oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,npd", [(256, 256), (256, 100), (257, 0), (257, 129), (257, 256), (258, 129)])
def test_rows_at_the_cap(n, npd):
    rng = np.random.default_rng(n + npd)
    q = rng.normal(size=(n, 3))
    q *= 2.6 * rng.uniform(0, 1, (n, 1)) ** (1 / 3) / np.linalg.norm(q, axis=1, keepdims=True)  # a ball of radius 2.6 A
    X = np.concatenate([q, np.full((n, 1), 0.1)], 1).reshape(-1)
    with A.FreeEntropy(npd, n - npd) as fe:
        fe.set_occupancy(np.full(n - npd, 0.3))
        if n > 257:
            with pytest.raises(A.A2CError) as e:
                fe.findNeighbors(X)
            assert e.value.code == A.A2C_ENBR_OVERFLOW
            return
        orc = O.Oracle(npd, n - npd, (0, 0, 0), (0, 0, 0), threads=8)
        assert orc.build_neighbors(X) == n - 1
        for _ in range(3):
            assert fe.findNeighbors(X)["max_neib"] == n - 1
            for w in ("PdPd", "PdH", "HPd", "HH", "HH1"):
                go, gi = fe.neighbors(w)
                oo, oi = orc.neighbors(w)
                assert np.array_equal(go, oo) and np.array_equal(gi, oi), w
            assert np.array_equal(fe.pdpdnum(), orc.pdpdnum())

"""Pair-once passes at the edges of their row order, lane units and tables,
against the oracle: species whose site counts leave every remainder modulo
four and straddle the 64-, 256- and 512-lane units, lanes per site 1..16,
both rules and precisions; and specimens whose quadrature nodes leave the
tables' [1, 6) A (wide packets), evaluated node by node.

Bars as elsewhere: FP64 objective 1e-10, gradient 1e-8 of its largest
component; mixed objective 1e-7, gradient 1e-5 in the 2-norm."""
import numpy as np
import pytest

import a2c_amd as A
import oracle as O
from helpers import specimen

pytestmark = pytest.mark.gpu


def cut(n, npd, nh, seed, sigma=(0.08, 0.15)):
    """npd Pd and nh H sites drawn from an n^3-cell specimen (free boundaries)."""
    X, x, box, per, p, h = specimen(n, seed=seed, disp=0.03, sigma=sigma, x=(0.01, 0.6), periodic=False)
    rng = np.random.default_rng(seed)
    ip = np.sort(rng.permutation(p)[:npd])
    ih = np.sort(rng.permutation(h)[:nh])
    X = X.reshape(-1, 4)
    return np.concatenate([X[ip], X[p + ih]]).reshape(-1), x[ih], box, per


def check(X, x, box, per, npd, nh, quad, lanes=None):
    try:
        if lanes:
            A.tune_set({"max_sites": [2**31 - 1], "lanes_mixed": [lanes], "lanes_fp64": [lanes]})
        orc = O.Oracle(npd, nh, box, per, T=400.0, threads=8, quad=quad)
        orc.build_neighbors(X)
        fo, Go = orc.eval(X, x)
        for prec in ("fp64", "mixed"):
            with A.FreeEntropy(npd, nh, box, per, T=400.0, precision=prec, quad=quad) as fe:
                fe.set_occupancy(x)
                fe.findNeighbors(X)
                for again in range(2):  # the second build refreshes from skin lists
                    f, G = fe.eval(X)
                    if prec == "fp64":
                        assert abs(f - fo) <= 1e-10 * abs(fo)
                        assert np.max(np.abs(G - Go)) <= 1e-8 * np.abs(Go).max()
                    else:
                        assert abs(f - fo) <= 1e-7 * abs(fo)
                        assert np.linalg.norm(G - Go) <= 1e-5 * np.linalg.norm(Go)
                    fe.findNeighbors(X)
    finally:
        A.tune_set(None)


@pytest.mark.parametrize("quad", ["r12", "gh3"])
@pytest.mark.parametrize("npd,nh", [(1, 0), (3, 5), (63, 65), (129, 254), (255, 257), (513, 511), (510, 1)])
def test_row_counts(npd, nh, quad):
    check(*cut(6, npd, nh, npd + nh), npd, nh, quad)


@pytest.mark.parametrize("lanes", [1, 2, 4, 8, 16])
def test_lanes_per_site(lanes):
    check(*cut(5, 257, 131, lanes), 257, 131, "r12", lanes)


@pytest.mark.parametrize("quad", ["r12", "gh3"])
def test_nodes_beyond_the_tables(quad):
    # Pd alone, nodes from 1.4 A up to 6.6 A (12-point) and 6.9 A (Gauss-Hermite): exponential tails
    check(*cut(4, 100, 0, 7, sigma=(0.30, 0.50) if quad == "r12" else (0.20, 0.35)), 100, 0, quad)


def test_wide_packets_gh3():
    # Pd-H nodes down to 1.1 A, Pd-Pd nodes beyond 6 A
    check(*cut(4, 100, 90, 7, sigma=(0.20, 0.35)), 100, 90, "gh3")


def test_nodes_below_the_tables():
    # packets that put Pd-H nodes under 1 A: closed forms in FP64, refused in mixed precision
    npd, nh = 100, 90
    X, x, box, per = cut(4, npd, nh, 7, sigma=(0.30, 0.50))
    orc = O.Oracle(npd, nh, box, per, T=400.0, threads=8)
    orc.build_neighbors(X)
    fo, Go = orc.eval(X, x)
    with A.FreeEntropy(npd, nh, box, per, T=400.0) as fe:
        fe.set_occupancy(x)
        fe.findNeighbors(X)
        f, G = fe.eval(X)
        assert abs(f - fo) <= 1e-10 * abs(fo)
        assert np.max(np.abs(G - Go)) <= 1e-8 * np.abs(Go).max()
        fe.set_precision("mixed")
        with pytest.raises(A.A2CError) as err:
            fe.eval(X)
        assert err.value.code == A.A2C_ENONFINITE

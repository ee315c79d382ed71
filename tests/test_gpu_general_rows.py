"""Pair-once passes of the general model at their edges, against the oracle:
site counts with every remainder modulo four and around the 64- and 256-lane
units, lanes per site 1..16, the smallest and largest node tables, tables that
end inside the cutoff, central differences, and the density in site order.

Bars as for the general model elsewhere: FP64 objective and densities to 1e-10,
gradient to 1e-8 of its largest component; mixed against FP64 1e-6 and 1e-4."""
import numpy as np
import pytest

import a2c_amd as A
import oracle as O
from helpers import product_rule_2pt, sampled_tables, specimen

pytestmark = pytest.mark.gpu


def cut(npd, nh, seed):
    """npd Pd and nh H sites drawn from a 5^3-cell specimen (free boundaries)."""
    X, x, box, per, p, h = specimen(5, seed=seed, disp=0.03, sigma=(0.08, 0.15), x=(0.01, 0.6), periodic=False)
    rng = np.random.default_rng(seed)
    ip, ih = np.sort(rng.permutation(p)[:npd]), np.sort(rng.permutation(h)[:nh])
    X = X.reshape(-1, 4)
    return np.concatenate([X[ip], X[p + ih]]).reshape(-1), x[ih], box, per


def many_nodes(K):
    """K nodes, swap-symmetric: pairs (a, b), (b, a) of random 3-vectors."""
    rng = np.random.default_rng(K)
    a, b = rng.normal(size=(2, K // 2, 3))
    xi = np.concatenate([np.concatenate([a, b], 1), np.concatenate([b, a], 1)])
    w = rng.uniform(0.5, 1.5, K // 2)
    w = np.concatenate([w, w])
    return xi, w / w.sum()


@pytest.mark.parametrize("npd,nh,lanes,quad,deriv,tables", [
    (1, 0, 1, None, "analytic", {}),
    (3, 5, 16, "one", "analytic", {}),
    (63, 66, 1, None, "fd", {}),
    (130, 255, 2, None, "analytic", {"n_r": 4501}),          # ends at 4.5 A
    (257, 129, 4, "product", "analytic", {"n_r": 2600, "d_r": 2e-3}),
    (259, 254, 8, "gh3", "analytic", {}),
    (40, 31, 2, "512", "analytic", {}),
    (40, 31, 16, "gh3", "fd", {}),
])
def test_edges(npd, nh, lanes, quad, deriv, tables):
    X, x, box, per = cut(npd, nh, npd + nh)
    one = O.Oracle(1, 0)  # the oracle's last potential answers O.eam: make it the closed forms
    one.build_neighbors(np.array([0.0, 0.0, 0.0, 0.1]))
    one.eval(np.array([0.0, 0.0, 0.0, 0.1]), np.zeros(0))
    t = sampled_tables(**tables)
    nodes = {"one": (np.zeros((1, 6)), np.ones(1)), "product": product_rule_2pt(), "512": many_nodes(512)}.get(quad)
    rule = "gh3" if quad == "gh3" else "r12"
    try:
        A.tune_set({"max_sites": [2**31 - 1], "lanes_mixed": [lanes], "lanes_fp64": [lanes]})
        O.set_tabulated(t)
        if nodes:
            O.set_quad_table(*nodes)
        orc = O.Oracle(npd, nh, box, per, T=400.0, deriv=deriv, threads=8, potential="tab",
                       quad="table" if nodes else rule)
        orc.build_neighbors(X)
        fo, Go = orc.eval(X, x)
        ro = orc.density(X, x)
        res = {}
        for prec in ("fp64", "mixed"):
            with A.FreeEntropy(npd, nh, box, per, T=400.0, deriv=deriv, precision=prec, quad=rule) as fe:
                fe.set_potential_tables(t)
                if nodes:
                    fe.set_quadrature(*nodes)
                fe.set_occupancy(x)
                fe.findNeighbors(X)
                fe.eval(X)
                rho = fe.density(X)  # leaves its arrays in site order; the next evaluation rewrites them
                res[prec] = fe.eval(X)
                assert np.max(np.abs(rho - ro)) <= 1e-10 * np.abs(ro).max()
        f, G = res["fp64"]
        assert abs(f - fo) <= 1e-10 * abs(fo)
        assert np.max(np.abs(G - Go)) <= 1e-8 * np.abs(Go).max()
        fm, Gm = res["mixed"]
        assert abs(fm - f) <= 1e-6 * abs(f)
        assert np.linalg.norm(Gm - G) <= 1e-4 * np.linalg.norm(G)
    finally:
        A.tune_set(None)

"""One pair alone in the FP64 evaluation, against the closed forms and the
quadrature rule in 50 digits: objective and gradient of two sites at distances
that put nodes on both sides of the forms' joints and of what the passes do
differently (f_H's tail beyond 5.35 A, the tables' last intervals, pairs with a
node past 6 A).

The bar: 2e-13 of the sum of the terms' magnitudes.  The functions are held to
~1e-15 of theirs (tests/test_pass_tables.py); F' and the sums add some hundred
roundings of 1.1e-16, and positions of a few A one of 4e-16 A, times slopes of
at most 5 per A."""
from decimal import Decimal

import numpy as np
import pytest

import a2c_amd as A
from eam_exact import D, F_H, F_PD, PHI_HH, PHI_PD, PHI_PDH, R_FUNCTIONS, Dual, embed_h, embed_pd

pytestmark = pytest.mark.gpu

KB = D(8.6173324e-5)
T, OCC = 400.0, (0.35, 0.6)
KINDS = {"PdPd": (0, 0), "PdH": (0, 1), "HH": (1, 1)}
# distance along a general direction, rc above all of them
DISTANCES = [1.8, 1.95, 2.2, 2.75, 3.9, 4.8, 4.98, 5.04, 5.2, 5.34, 5.6, 5.9]
SIGMA = (0.11, 0.08)


def nodes(rule, d, s):
    """(weight, vector) of the rule's nodes for pair vector d = q_0 - q_1"""
    if rule == "r12":
        six = Dual(Decimal(6).sqrt())
        for end in (0, 1):
            for c in range(3):
                for sign in (1, -1):
                    yield Decimal(1) / 12, [d[k] + (six * s[end] * float(sign if end == 0 else -sign) if k == c else 0.0)
                                            for k in range(3)]
    else:
        w = {0: Decimal(2) / 3, 1: Decimal(1) / 6, -1: Decimal(1) / 6}
        sd = (s[0] * s[0] + s[1] * s[1]).sqrt() * Dual(Decimal(3).sqrt())
        for a in (-1, 0, 1):
            for b in (-1, 0, 1):
                for c in (-1, 0, 1):
                    yield w[a] * w[b] * w[c], [d[k] + sd * float(z) for k, z in enumerate((a, b, c))]


def objective(kind, rule, X, dx):
    """f of the pair and its derivative along dx, and the sums of magnitudes"""
    q = [Dual(D(v), Decimal(t)) for v, t in zip(X, dx)]
    sp = KINDS[kind]
    occ = [D(OCC[k]) if sp[k] else Decimal(1) for k in (0, 1)]
    dens = [F_H if s else F_PD for s in sp]
    phi = {(0, 0): PHI_PD, (0, 1): PHI_PDH, (1, 1): PHI_HH}[sp]
    rho, pair, mag, dmag = [Dual(0.0), Dual(0.0)], Dual(0.0), Decimal(0), Decimal(0)
    for w, r in nodes(rule, [q[k] - q[4 + k] for k in range(3)], (q[3], q[7])):
        rn = (r[0] * r[0] + r[1] * r[1] + r[2] * r[2]).sqrt()
        f = {fn: R_FUNCTIONS[fn](rn) for fn in {dens[0], dens[1], phi}}
        for k in (0, 1):  # the density at k comes from the other site
            rho[k] = rho[k] + f[dens[1 - k]] * Dual(w * occ[1 - k])
        pair = pair + f[phi] * Dual(w * occ[0] * occ[1])
        mag += w * abs(f[phi].v)
        dmag += w * (abs(f[phi].d) + sum(abs(f[x].d) for x in dens))
    V, ent = pair, Dual(0.0)
    for k in (0, 1):
        F = embed_h(rho[k]) if sp[k] else embed_pd(rho[k])
        V = V + F * Dual(occ[k])
        mag += abs(F.v)
        ent = ent + q[4 * k + 3].log() * Dual(3 * KB * occ[k])
        dmag += 3 * KB * occ[k] * D(T) * abs(q[4 * k + 3].d / q[4 * k + 3].v)
    f = V * Dual(1 / D(T)) - ent
    return f, float(mag / D(T) + abs(ent.v)), float(dmag / D(T))


@pytest.mark.parametrize("rule", ["r12", "gh3"])
@pytest.mark.parametrize("kind", list(KINDS))
def test_one_pair(kind, rule):
    direction = np.array([0.48, -0.6, 0.64])
    sp = KINDS[kind]
    npd = 2 - sum(sp)
    with A.FreeEntropy(npd, 2 - npd, (0, 0, 0), (0, 0, 0), T=T, rc=6.2, quad=rule) as fe:
        fe.set_occupancy(np.array([OCC[k] for k in (0, 1) if sp[k]]))
        for dist in DISTANCES:
            X = np.concatenate([dist * direction, [SIGMA[0]], [0.0, 0.0, 0.0, SIGMA[1]]])
            fe.findNeighbors(X)
            f, G = fe.formFunctionAndGradient(X)
            for c in range(8):
                want, mag, dmag = objective(kind, rule, X, np.eye(8)[c])
                if c == 0:
                    assert abs(float(D(f) - want.v)) <= 2e-13 * mag, (dist, f, float(want.v), mag)
                assert abs(float(D(G[c]) - want.d)) <= 2e-13 * dmag, (dist, c, G[c], float(want.d), dmag)

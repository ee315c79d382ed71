"""The tables that the pair-once passes read, each evaluated on the host as the
kernels do it (a2c_eam_pass), against the closed forms in 50 digits over [1, 6) A.

The bars, per interval of r, allow what the passes' arithmetic rounds, U (|y| + r
|y'|) with U = 16 2^-53 in FP64 (a Horner scheme of degree 8 for value and slope)
and 2 2^-24 in the mixed passes, and beyond it no more error than the plainer method has on the same interval: the tables in r of
high degree (a2c_eam_tables64: f_H, phi_PdH, phi_HH) and the Hermite tables in
r (a2c_eam_tables); for the Pd functions in FP64, whose closed forms are products
that cancel, 1/512 of what these lose in FP64 (the tables are built from the same
products in 80 bits, 2,048 times as fine)."""
from decimal import Decimal

import numpy as np
import pytest

import a2c_amd as A
import oracle as O
from eam_exact import D, F_H, F_PD, PHI_HH, PHI_PD, PHI_PDH, R_FUNCTIONS, Dual

ORACLE = [O.RHO_PD, O.RHO_H, O.PHI_PD, O.PHI_PDH, O.PHI_H]
EDGES = [1.0, 1.1, 1.2, 1.4, 1.6, 1.8, 2.0, 2.25, 2.5, 3.0, 3.5, 4.0, 4.5, 4.9, 5.0, 5.05, 5.1, 5.2, 5.34, 5.35,
         5.36, 5.5, 5.99]
SWITCH = np.array([5.0, 5.05, 5.35])


def exact(fn, r):
    out = [R_FUNCTIONS[fn](Dual(D(x), Decimal(1))) for x in r]
    return [(y.v, y.d) for y in out]


def error(got, want):
    return np.array([abs(float(D(g) - w)) for g, w in zip(got, want)])


def horner(c, u, h):
    v = np.zeros_like(u)
    d = np.zeros_like(u)
    for j in range(c.shape[1] - 1, -1, -1):
        d = d * u + v
        v = v * u + c[:, j]
    return v, d / h


def plain(fn, r, precision):
    """values and slopes of the plainer method"""
    if precision == "mixed":
        tab = A.eam_tables().astype(np.float64)
        h = 5.0 / tab.shape[1]
        k = np.floor((r - 1.0) / h).astype(int)
        return horner(tab[fn, k], (r - 1.0) / h - k, h)
    if fn in (F_PD, PHI_PD):
        return O.eam(ORACLE[fn], r), O.eam_d(ORACLE[fn], r)
    tab = A.eam_tables64()[0][{F_H: 0, PHI_PDH: 1, PHI_HH: 2}[fn]][:, :9]
    k = np.floor((r - 1.0) / 0.05).astype(int)
    return horner(tab[k], (r - 1.0) / 0.05 - k, 0.05)


CASES = [(p, f) for p in ("fp64", "mixed") for f in range(5)]


@pytest.mark.parametrize("precision,fn", CASES)
def test_pass_tables(precision, fn):
    rng = np.random.default_rng(fn)
    unit = 16 * 2.0 ** -53 if precision == "fp64" else 2 * 2.0 ** -24
    bad = []
    for lo, hi in zip(EDGES[:-1], EDGES[1:]):
        r = rng.uniform(lo, hi, 48)
        r = r[np.min(np.abs(r[:, None] - SWITCH), axis=1) > (1e-9 if precision == "fp64" else 2e-6)]
        at, v, d = A.eam_pass(fn, r, precision)
        want = exact(fn, at)
        ev, ed = error(v, [w[0] for w in want]), error(d, [w[1] for w in want])
        pv, pd = plain(fn, at, precision)
        share = 512.0 if precision == "fp64" and fn in (F_PD, PHI_PD) else 1.0
        if precision == "mixed" and fn == F_H:  # evaluated without a table: rounding alone
            share = np.inf
        rv = np.max(error(pv, [w[0] for w in want])) / share
        rd = np.max(error(pd, [w[1] for w in want])) / share
        slope = np.abs([float(w[1]) for w in want])
        value = np.abs([float(w[0]) for w in want])
        curve = np.abs(O.eam_d(ORACLE[fn], at * (1 + 1e-5)) - O.eam_d(ORACLE[fn], at * (1 - 1e-5))) / (2e-5 * at)
        bv = unit * (value + at * slope) + rv
        bd = unit * (slope + at * curve) + rd
        if np.any(ev > bv) or np.any(ed > bd):
            bad.append((lo, hi, "value %.1e of %.1e" % (ev[np.argmax(ev / bv)], bv[np.argmax(ev / bv)]),
                        "slope %.1e of %.1e" % (ed[np.argmax(ed / bd)], bd[np.argmax(ed / bd)])))
    assert not bad, "\n".join(map(str, bad))


@pytest.mark.parametrize("fn", [PHI_PDH, PHI_HH])
@pytest.mark.parametrize("lo,hi", [(1.7, 2.2), (2.2, 2.6), (3.2, 3.6), (4.2, 4.6)])
def test_mixed_coordinate_noise(fn, lo, hi):
    """What a pair function's value in the mixed passes loses to its argument: the
    rms error over the slope is at most half an FP32 unit of r (two roundings of rms
    0.29 units beside the table coordinate's), plus one of the value.  Noise of the
    objective ends the mixed phase of a relaxation; a rounded radius alone leaves
    0.8 units."""
    r = np.random.default_rng(fn).uniform(lo, hi, 20000)
    at, v, _ = A.eam_pass(fn, r, "mixed")
    e, slope = O.eam(ORACLE[fn], at), np.mean(np.abs(O.eam_d(ORACLE[fn], at)))
    rms = np.sqrt(np.mean((v - e) ** 2)) / slope
    assert rms <= 2.0 ** -24 * (0.5 * np.mean(r) + np.mean(np.abs(e)) / slope)

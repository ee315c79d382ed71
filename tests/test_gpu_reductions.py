"""Sums by the last block to arrive, at the edges of their blocks of 256 sites:
relaxations of one to three blocks, alone and in one batch with others and an
empty lattice, in the vector-free and the per-step form of the recursion.

Both forms build the same directions up to the rounding of their sums, so six
FP64 iterations agree to 1e-9 in f (relative) and 1e-7 A in X; a lattice's
results do not depend on the batch it is in, bit for bit."""
import os

import numpy as np
import pytest

import a2c_amd as A
from helpers import specimen

pytestmark = pytest.mark.gpu

SIZES = (2, 255, 256, 257, 513, 600, 0)


def cut(n):
    X, x, box, per, p, h = specimen(6, seed=n, disp=0.02, sigma=(0.09, 0.12), x=(0.05, 0.6), periodic=False)
    npd = (n + 1) // 2
    X = X.reshape(-1, 4)
    return np.concatenate([X[:npd], X[p:p + n - npd]]).reshape(-1), x[:n - npd], box, per, npd, n - npd


def relax(sizes, form):
    old = os.environ.get("A2C_TWO_LOOP")
    os.environ["A2C_TWO_LOOP"] = form
    try:
        b = A.Batch(precision="fp64", max_lattices=len(sizes))
    finally:
        os.environ.pop("A2C_TWO_LOOP")
        if old is not None:
            os.environ["A2C_TWO_LOOP"] = old
    slots = []
    for n in sizes:
        X, x, box, per, npd, nh = cut(n)
        slots.append(b.add(X, x, npd, nh, box, per, T=400.0))
        b.start(slots[-1], max_it=6)
    while b.step(6):
        pass
    return {n: (b.report(s), b.get_state(s)[0]) for n, s in zip(sizes, slots)}


def test_blocks():
    vf, ps = relax(SIZES, ""), relax(SIZES, "perstep,segmented")
    assert vf[0][0]["gnorm"] == 0.0 and vf[0][0]["f"] == 0.0
    for n in SIZES[:-1]:
        (r, X), (q, Y) = vf[n], ps[n]
        assert r["iterations"] == q["iterations"]
        assert abs(r["f"] - q["f"]) <= 1e-9 * abs(q["f"])
        assert np.max(np.abs(X - Y)) <= 1e-7
        ra, Xa = relax((n,), "")[n]
        assert ra["f"] == r["f"] and np.array_equal(Xa, X)


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
@pytest.mark.parametrize("first", [1, 6, 400])
def test_a_slot_relaxes_again_as_the_first_time(precision, first):
    """A relaxation leaves nothing to the next one of its slot: stopped after
    `first` iterations or converged, a new start from the same state gives the
    same report and state, bit for bit."""
    X, x, box, per, npd, nh = cut(513)
    with A.Batch(precision=precision, max_lattices=1) as b:
        s = b.add(X, x, npd, nh, box, per, T=400.0)
        runs = []
        for it in (first, 400, 400):
            b.set_state(s, X)
            b.start(s, max_it=it)
            while b.step(7):
                pass
            runs.append((b.report(s), b.get_state(s)[0]))
    assert runs[1][0] == runs[2][0] and np.array_equal(runs[1][1], runs[2][1])
    if first == 400:
        assert runs[0][0] == runs[1][0] and np.array_equal(runs[0][1], runs[1][1])

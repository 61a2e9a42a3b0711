"""Generators of one workgroup (a row per thread) at every register width: rows of 1
to 17 and more entries, an odd number of rows, one wavefront and the most rows of
each kernel, against the oracle and against the stage kernels."""
import numpy as np
import pytest

import oracle
import quac_amd as qa
import recipes
from qbuild import build_system

pytestmark = pytest.mark.gpu


def _coupled(dims):
    terms = []
    for s, n in enumerate(dims):
        terms += [("ham", 0.3 + 0.1 * s, [(s, "n")]), ("ham", 0.2, [(s, "lower")]), ("ham", 0.2, [(s, "raise")]),
                  ("lin", 0.05, [(s, "lower")])]
    return {"subs": [("op", n) for n in dims], "terms": terms, "mcwf": False}


def _start(n):
    rng = np.random.default_rng(11)
    psi = rng.normal(size=n) + 1j * rng.normal(size=n)
    return np.outer(psi.conj(), psi).reshape(-1) / np.linalg.norm(psi) ** 2


# entries of the longest row: 1, 5, 6 (one ladder), 11 (two), 16 (three), 21 (four)
@pytest.mark.parametrize("recipe", [
    {"subs": [("op", 3)], "terms": [("ham", 1.0, [(0, "n")]), ("lin", 0.1, [(0, "n")])], "mcwf": False},
    recipes.jc_recipe(levels=14), _coupled((2,)), _coupled((25,)), _coupled((28,)), _coupled((4, 6)), _coupled((4, 7)),
    _coupled((2, 3, 4)), _coupled((2, 2, 2, 2)),
], ids=["diagonal", "jc", "2", "25", "28", "4x6", "4x7", "2x3x4", "2x2x2x2"])
def test_small_generators(recipe):
    qs, _, _ = build_system(recipe)
    A = qs.matrix()
    tot, terms = recipes.oracle_terms(recipe)
    x0, dt, steps = _start(tot), 0.02, 7
    ref = oracle.construct(tot, terms, dm=True).rk4(x0, dt, steps)
    rp, _, val = A.export()
    norm = np.add.reduceat(np.abs(np.append(val, 0)), rp[:-1]).max()
    for prec, eps in ((qa.FP64, 2.0 ** -53), (qa.FP32, 2.0 ** -47)):
        v = qa.DeviceVec(tot * tot, prec)
        v.set(x0)
        qa.rk4_device(A, v, dt, steps)
        # a few roundings of the state and of h A times it per step
        assert np.abs(v.get() - ref).max() <= (steps * (2 * dt * norm + 8) + 1) * np.abs(x0).max() * eps
    qs.destroy()


def _bogacki_shampine(f, x, t1, h):
    """the integrator in numpy: tolerances 5e-7, the next step 0.9 err^(-1/3) times the
    last within [0.1, 10], kept in [0.01, 1]"""
    t, k1, steps, eps = 0.0, None, 0, 1e-12 * (t1 + h + 1.0)
    while t < t1 - eps:
        hh = min(h, t1 - t)
        k1 = f(x) if k1 is None else k1
        k2 = f(x + hh / 2 * k1)
        k3 = f(x + 3 * hh / 4 * k2)
        xn = x + hh * (2 / 9 * k1 + 1 / 3 * k2 + 4 / 9 * k3)
        k4 = f(xn)
        e = hh * ((2 / 9 - 7 / 24) * k1 + (1 / 3 - 1 / 4) * k2 + (4 / 9 - 1 / 3) * k3 - 1 / 8 * k4)
        err = np.sqrt(np.mean((np.abs(e) / (5e-7 + 5e-7 * np.maximum(np.abs(x), np.abs(xn)))) ** 2))
        h = min(1.0, max(0.01, hh * min(10.0, max(0.1, 0.9 * err ** (-1 / 3)))))
        if err <= 1.0 or hh <= 0.01 * (1 + 1e-12):
            x, k1, t, steps = xn, k4, t + hh, steps + 1
    return x, steps


@pytest.mark.parametrize("dims", [(2,), (5,), (25,), (4, 6), (2, 3, 4), (2, 2, 2, 3)])
def test_small_adaptive_matches_numpy(dims):
    r = _coupled(dims)
    qs, _, _ = build_system(r)
    tot, _ = recipes.oracle_terms(r)
    x0 = _start(tot)
    qa.set_option("ts_rk_type", "3bs")
    qa.set_option("ts_adapt_type", "basic")
    x = qs.create_qvec()
    x.set(x0)
    steps, t = qs.time_step(x, 0.0, 1.0, 0.01, 10 ** 6)
    qa.set_option("ts_rk_type", "4")
    qa.set_option("ts_adapt_type", "none")
    rp, col, val = qs.matrix().export()
    rows = np.repeat(np.arange(tot * tot), np.diff(rp))

    def f(v):
        p = val * v[col]
        return (np.bincount(rows, p.real, tot * tot) + 1j * np.bincount(rows, p.imag, tot * tot))

    ref, ref_steps = _bogacki_shampine(f, x0, 1.0, 0.01)
    assert abs(t - 1.0) < 1e-9 and steps == ref_steps
    # roundings of the state and of h A times it in every step (h <= 1), and of the step
    # sizes, which move the state by their relative error times h A
    norm = np.add.reduceat(np.abs(val), rp[:-1]).max()
    assert np.abs(x.get() - ref).max() <= steps * (4 * norm + 8) * np.abs(x0).max() * 2.0 ** -53
    x.destroy()
    qs.destroy()


def _wide(dims, exchange, squeezed=()):
    r = _coupled(dims)
    for a, b in exchange:
        r["terms"] += [("ham", 0.1, [(a, "raise"), (b, "lower")]), ("ham", 0.1, [(b, "raise"), (a, "lower")])]
    for a, b in squeezed:
        r["terms"] += [("ham", 0.07, [(a, "raise"), (b, "raise")]), ("ham", 0.07, [(a, "lower"), (b, "lower")])]
    return r


RING = [(0, 1), (1, 2), (0, 2)]


# the entries off the diagonal of the longest row: every width of the kernels for up to
# 640 rows and for up to 800
@pytest.mark.parametrize("recipe,off", [
    (_coupled((3, 9)), 10), (_wide((4, 6), [(0, 1)]), 14), (_wide((4, 7), [(0, 1)]), 14),
    (_wide((4, 6), [(0, 1)], [(1, 1)]), 18), (_wide((4, 7), [(0, 1)], [(1, 1)]), 18),
    (_wide((3, 3, 3), [(0, 1), (1, 2)]), 23), (_wide((2, 3, 4), RING, [(1, 2)]), 25),
    (_wide((2, 3, 4), RING, RING), 29), (_wide((3, 3, 3), RING, [(0, 1)]), 31), (_wide((3, 3, 3), RING, RING), 39),
])
def test_wide_rows(recipe, off):
    qs, _, _ = build_system(recipe)
    A = qs.matrix()
    tot, terms = recipes.oracle_terms(recipe)
    x0, dt, steps = _start(tot), 0.02, 7
    ref = oracle.construct(tot, terms, dm=True).rk4(x0, dt, steps)
    rp, col, val = A.export()
    rows = np.repeat(np.arange(tot * tot), np.diff(rp))
    assert np.bincount(rows[col != rows]).max() == off
    norm = np.add.reduceat(np.abs(val), rp[:-1]).max()
    for prec, eps in ((qa.FP64, 2.0 ** -53), (qa.FP32, 2.0 ** -47)):
        v = qa.DeviceVec(tot * tot, prec)
        v.set(x0)
        qa.rk4_device(A, v, dt, steps)
        # a few roundings of the state and of h A times it per step
        assert np.abs(v.get() - ref).max() <= (steps * (2 * dt * norm + 8) + 1) * np.abs(x0).max() * eps
    qs.destroy()

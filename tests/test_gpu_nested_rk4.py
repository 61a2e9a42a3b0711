"""The nested form of the RK4 step of a constant generator (four launches of
y = x + c A y', qh_spmv.hip / qh_ks2.hip) on every kernel variant, at row counts
with a remainder in each tile (64-row and 128-row slices, 2048-row windows, an odd
last row), against the oracle's classic RK4 in FP64."""
import ctypes

import numpy as np
import pytest

import oracle
import quac_amd as qa
import recipes
from qbuild import build_system

pytestmark = pytest.mark.gpu


def _recipe(dims):
    """coupled ladders with decay: every subsystem driven and damped"""
    terms = []
    for s, n in enumerate(dims):
        terms += [("ham", 0.3 + 0.1 * s, [(s, "n")]), ("ham", 0.2, [(s, "lower")]), ("ham", 0.2, [(s, "raise")]),
                  ("lin", 0.05, [(s, "lower")]), ("lin", 0.02, [(s, "n")])]
    for s in range(len(dims) - 1):
        terms += [("ham", 0.15, [(s, "raise"), (s + 1, "lower")]), ("ham", 0.15, [(s + 1, "raise"), (s, "lower")])]
    return {"subs": [("op", n) for n in dims], "terms": terms, "mcwf": False}


@pytest.mark.parametrize("dims", [(3, 5), (2, 4, 4), (3, 3, 5), (7, 7)])
@pytest.mark.parametrize("lanes", [1, 8, 64, 128, 130, 132, 134, 136, 140, 141, 142, 143, 144])
def test_nested_rk4_matches_oracle(dims, lanes):
    r = _recipe(dims)
    qs, _, _ = build_system(r)
    A = qs.matrix()
    N = int(np.prod(dims))
    rng = np.random.default_rng(3)
    psi = rng.normal(size=N) + 1j * rng.normal(size=N)
    psi /= np.linalg.norm(psi)
    x0 = np.outer(psi.conj(), psi).reshape(-1)
    tot, terms = recipes.oracle_terms(r)
    steps, dt = 11, 0.02  # a graph of 8 steps and 3 launched by themselves
    ref = oracle.construct(tot, terms, dm=True).rk4(x0, dt, steps)
    rp, _, val = A.export()
    norm = max(np.abs(val[rp[i]:rp[i + 1]]).sum() for i in range(N * N))
    big = np.abs(x0).max()
    for prec in (qa.FP64, qa.FP32):
        if prec == qa.FP64 and lanes >= 140:
            continue
        A.set_lanes(lanes if lanes < 140 else 8, lanes)
        v = qa.DeviceVec(N * N, prec)
        v.set(x0)
        qa.rk4_device(A, v, dt, steps)
        # per step: the rounding of the stored values and of the last stage's input
        # (2^-24 of each product in FP32), h |A| of the state at most, and a few
        # roundings of the state itself in FP64
        eps = 2.0 ** -24 if prec == qa.FP32 else 2.0 ** -53
        tol = steps * big * (2 * dt * norm * eps + 8 * 2.0 ** -48)
        if prec == qa.FP64:
            tol = steps * big * (2 * dt * norm + 8) * eps
        assert np.abs(v.get() - ref).max() <= tol, (lanes, prec)
    A.set_lanes(0, 0)
    qs.destroy()


@pytest.mark.parametrize("dims", [(2, 4, 4), (7, 7)])
@pytest.mark.parametrize("lanes", [129, 131, 133, 135, 137, 138, 145, 146])
def test_nested_rk4_other_variants(dims, lanes):
    """the remaining variants, among them those that hold a slice's slot metadata in
    registers"""
    test_nested_rk4_matches_oracle(dims, lanes)


@pytest.mark.parametrize("lanes", [133, 134, 137, 138, 140, 143, 145, 146])
def test_metadata_of_long_slices(lanes):
    """entries without order, so that nearly every one is a slot of its own and a slice has
    more than 64: the variants that hold the metadata in registers read it from memory"""
    n, w, dt = 1100, 4, 0.01
    rng = np.random.default_rng(4)
    col = np.sort(np.array([rng.choice(n, w, replace=False) for _ in range(n)]), axis=1).astype(np.int64)
    val = rng.normal(size=(n, w)) + 1j * rng.normal(size=(n, w))
    rp = (w * np.arange(n + 1)).astype(np.int64)
    h = ctypes.c_void_p()
    assert qa.lib().qh_mat_from_csr(ctypes.c_int64(n), *[a.ctypes.data_as(ctypes.c_void_p) for a in (rp, col, val)],
                                    ctypes.byref(h)) == 0
    A = qa.Matrix(h, owned=True)
    prec = qa.FP32 if lanes >= 140 else qa.FP64
    lay = A.pair_layout_info() if lanes >= 140 else A.layout_info()
    assert lay["slots"] > 64 * lay["slices"]
    A.set_lanes(lanes if lanes < 140 else 8, lanes)
    x0 = rng.normal(size=n) + 1j * rng.normal(size=n)
    v = qa.DeviceVec(n, prec)
    v.set(x0)
    qa.rk4_device(A, v, dt, 3)
    ref = x0
    for _ in range(3):
        y = ref
        for c in (dt / 4, dt / 3, dt / 2, dt):
            y = ref + c * (val * y[col]).sum(axis=1)
        ref = y
    norm = np.abs(val).sum(axis=1).max()
    eps = 2.0 ** -24 if prec == qa.FP32 else 2.0 ** -53
    tol = 3 * np.abs(x0).max() * (2 * dt * norm * eps + 8 * (2.0 ** -48 if prec == qa.FP32 else eps))
    assert np.abs(v.get() - ref).max() <= tol

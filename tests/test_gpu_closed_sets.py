"""RK4 of generators whose rows fall apart into closed sets (qh_comp.hip), one set or
several per workgroup, against the oracle's classic RK4 in FP64 and against the stage
kernels that a forced variant selects: one and two rows a thread, entries in
registers and in memory, slices with a remainder, real, imaginary and complex
entries, rows without entries, uneven blocks of a batch."""
import numpy as np
import pytest

import oracle
import quac_amd as qa
import recipes
from qbuild import build_system

pytestmark = pytest.mark.gpu


def _tc(qubits, levels):
    """emitters and a cavity: excitation numbers split the rows"""
    c, terms = qubits, [("ham", 0.3, [(qubits, "n")])]
    for i in range(qubits):
        terms += [("ham", 0.1 + 0.02 * i, [(i, "raise"), (c, "lower")]), ("ham", 0.1 + 0.02 * i, [(c, "raise"), (i, "lower")])]
        terms += [("lin", 0.02, [(i, "lower")])]
    return {"subs": [("op", 2)] * qubits + [("op", levels)], "terms": terms + [("lin", 0.01, [(c, "lower")])], "mcwf": False}


def _noisy(qubits, extra=()):
    terms = [("lin", 0.02 + 0.01 * i, [(i, "lower")]) for i in range(qubits)]
    terms += [("lin", 0.03, [(i, "sz")]) for i in range(qubits)]
    return {"subs": [("op", 2)] * qubits, "terms": terms + list(extra), "mcwf": False}


def _diagonal(levels):
    """no off-diagonal entry: every row is a set"""
    return {"subs": [("op", levels)], "terms": [("ham", 0.7, [(0, "n")]), ("lin", 0.05, [(0, "n")])], "mcwf": False}


CASES = [
    _tc(1, 15),  # bins of 1 to 2 slices
    _tc(2, 9),
    _tc(3, 17),  # a component of 1028 rows: two rows a thread
    _noisy(6),
    _noisy(7),  # 16 384 rows, the most whose plan one workgroup forms
    _noisy(8),  # more bins than two a CU: bins of several components, a launch per shape
    _noisy(5, [("ham", 0.3, [(0, "sx")]), ("ham", 0.2, [(1, "sy")])]),  # real and imaginary entries
    _diagonal(31),
]


def _start(n):
    rng = np.random.default_rng(5)
    psi = rng.normal(size=n) + 1j * rng.normal(size=n)
    return np.outer(psi.conj(), psi).reshape(-1) / np.linalg.norm(psi) ** 2


def _steps(A, x0, prec, dt, steps, **kw):
    v = qa.DeviceVec(len(x0), prec)
    v.set(x0)
    qa.rk4_prepare(A, v, dt, **kw)  # the plan is formed now, whatever the steps
    qa.rk4_device(A, v, dt, steps, **kw)
    return v.get()


@pytest.mark.parametrize("recipe", CASES, ids=[str([n for _, n in c["subs"]]) for c in CASES])
def test_closed_sets_match_oracle(recipe):
    qs, _, _ = build_system(recipe)
    A = qs.matrix()
    tot, terms = recipes.oracle_terms(recipe)
    x0, dt = _start(tot), 0.02
    m = oracle.construct(tot, terms, dm=True)
    rp, _, val = A.export()
    norm = np.add.reduceat(np.abs(np.append(val, 0)), rp[:-1]).max() if len(val) else 0.0
    for steps in (1, 7):
        ref = m.rk4(x0, dt, steps)
        for prec in (qa.FP64, qa.FP32):
            # a few roundings of the state and of h A times it per step; FP32: the state
            # is kept as two words, the generator in 64 bits
            eps = 2.0 ** -53 if prec == qa.FP64 else 2.0 ** -47
            tol = steps * np.abs(x0).max() * (2 * dt * norm + 8) * eps + (2.0 ** -47 if prec == qa.FP32 else 0.0)
            got = _steps(A, x0, prec, dt, steps)
            assert np.abs(got - ref).max() <= tol, (steps, prec)
            assert A.closed_info(prec)["bins"] > 0 or A.info()[0] <= 800
    A.set_lanes(8, 8)  # the stage kernels
    ref = _steps(A, x0, qa.FP64, dt, 7)
    A.set_lanes(0, 0)
    assert np.abs(_steps(A, x0, qa.FP64, dt, 7) - ref).max() <= 7 * np.abs(x0).max() * (2 * dt * norm + 8) * 2.0 ** -52
    qs.destroy()


def test_largest_sets_in_registers():
    """a component of 2048 rows and 11 slots: the most rows and slots of two rows a
    thread"""
    r = _noisy(11)
    qs, _, _ = build_system(r)
    A = qs.matrix()
    x0 = _start(2048)
    got = _steps(A, x0, qa.FP64, 0.02, 3)
    assert A.closed_info()["bins"] > 0 and A.closed_info()["word_bins"] == 0
    A.set_lanes(8, 0)
    ref = _steps(A, x0, qa.FP64, 0.02, 3)
    # rows of h A sum to at most 0.02 * 2 * 11 * 0.2 here
    assert np.abs(got - ref).max() <= 3 * np.abs(x0).max() * 16 * 2.0 ** -53
    qs.destroy()


# the largest set of four emitters and a cavity of n levels has 256 n - 280 rows: 2280 for
# 10 levels, 4584 and 4840 for 19 and 20 (the limit in FP64 is 4800), 7912 and 8168 for 32
# and 33 (8128 in FP32)
@pytest.mark.parametrize("levels,count,prec,words", [
    (10, 20, qa.FP32, True), (10, 20, qa.FP64, True), (19, 12, qa.FP64, True), (20, 12, qa.FP64, False),
    (32, 12, qa.FP32, True), (33, 12, qa.FP32, False)])
def test_entries_read_as_words(levels, count, prec, words):
    """components too large for registers, of up to 13 slots (more than are fetched
    ahead), enough of them to fill the chip; complex64 stage vectors in FP32"""
    recipe, dt, steps = _tc(4, levels), 0.02, 3
    systems = [build_system(recipe)[0] for _ in range(count)]
    n = 16 * levels
    b = qa.Batch([s.matrix() for s in systems], [n] * count, prec=prec)
    x0 = _start(n)
    for i in range(count):
        b.set_state(i, x0 if i % 2 else x0.conj())
    qa.rk4_prepare(b.matrix(), b.state(), dt)
    b.rk4(dt, steps)
    info = b.matrix().closed_info(prec)
    assert (info["word_bins"] > 0) == words and (info["bins"] > 0) == words
    tot, terms = recipes.oracle_terms(recipe)
    m = oracle.construct(tot, terms, dm=True)
    rp, _, val = systems[0].matrix().export()
    norm = np.add.reduceat(np.abs(val), rp[:-1]).max()
    # per step: h |A| of a state rounded to 32 bits, and the two words' rounding; FP64: a
    # few roundings of the state and of h A times it
    eps = (2 * dt * norm + 8) * 2.0 ** -53 if prec == qa.FP64 else 2 * dt * norm * 2.0 ** -24 + 8 * 2.0 ** -48
    for i in (0, count - 1):
        ref = m.rk4(x0 if i % 2 else x0.conj(), dt, steps)
        assert np.abs(b.get_state(i) - ref).max() <= steps * np.abs(x0).max() * eps
    if words:  # (the order of a row's slots on the sliced layout depends on where its block starts)
        assert np.array_equal(b.get_state(1), b.get_state(count - 1))
    b.destroy()
    for s in systems:
        s.destroy()


def test_renormalised_and_split_calls():
    """a call's steps are the same in one call or several, and the trace is restored
    every renorm_every steps"""
    r = _tc(2, 12)
    qs, _, _ = build_system(r)
    A = qs.matrix()
    x0 = _start(48)
    one = _steps(A, x0, qa.FP64, 0.01, 9)
    v = qa.DeviceVec(len(x0), qa.FP64)
    v.set(x0)
    for k in (1, 3, 5):
        qa.rk4_device(A, v, 0.01, k)
    assert np.array_equal(v.get(), one)
    f = _steps(A, 1.5 * x0, qa.FP32, 0.01, 10, tot=48, renorm_every=10)
    assert abs(np.trace(f.reshape(48, 48)) - 1.0) < 1e-12
    qs.destroy()


def test_batch_of_uneven_blocks():
    sizes = [(1, 7), (2, 11), (1, 2), (3, 9)]
    systems = [build_system(_tc(*s))[0] for s in sizes]
    tots = [2 ** q * n for q, n in sizes]
    b = qa.Batch([s.matrix() for s in systems], tots, prec=qa.FP64)
    starts = [_start(t) for t in tots]
    for i, x0 in enumerate(starts):
        b.set_state(i, x0)
    qa.rk4_prepare(b.matrix(), b.state(), 0.01)
    b.rk4(0.01, 6)
    assert b.matrix().closed_info()["bins"] > 0
    for i, (s, x0) in enumerate(zip(sizes, starts)):
        tot, terms = recipes.oracle_terms(_tc(*s))
        ref = oracle.construct(tot, terms, dm=True).rk4(x0, 0.01, 6)
        assert np.abs(b.get_state(i) - ref).max() <= 6 * 16 * 2.0 ** -53
    b.destroy()
    for s in systems:
        s.destroy()


@pytest.mark.parametrize("prec", [qa.FP64, qa.FP32])
@pytest.mark.parametrize("sizes", [[(3, 17), (4, 5)], [(3, 20), (4, 6), (2, 10)]])
def test_batch_of_shapes_with_no_common_kernel(sizes, prec):
    """three emitters of 17 or more levels (bins of more than 1024 rows and 10 slots)
    beside four emitters (up to 16 slots): a launch for every shape, and in the second
    batch bins that read their entries as words"""
    dt, steps = 0.01, 4
    systems = [build_system(_tc(*s))[0] for s in sizes]
    tots = [2 ** q * n for q, n in sizes]
    b = qa.Batch([s.matrix() for s in systems], tots, prec=prec)
    starts = [_start(t) for t in tots]
    for i, x0 in enumerate(starts):
        b.set_state(i, x0)
    qa.rk4_prepare(b.matrix(), b.state(), dt)
    b.rk4(dt, 1)
    b.rk4(dt, steps - 1)
    info = b.matrix().closed_info(prec)
    assert info["launches"] > 1 and (info["word_bins"] > 0) == (len(sizes) == 3)
    for i, (s, x0) in enumerate(zip(sizes, starts)):
        tot, terms = recipes.oracle_terms(_tc(*s))
        m = oracle.construct(tot, terms, dm=True)
        rp, _, val = systems[i].matrix().export()
        norm = np.add.reduceat(np.abs(val), rp[:-1]).max()
        # per step: a few roundings of the state and of h A times it; FP32 words: h |A| of
        # a state rounded to 32 bits, and the two words' rounding
        eps = (2 * dt * norm + 8) * 2.0 ** -53 if prec == qa.FP64 else 2 * dt * norm * 2.0 ** -24 + 8 * 2.0 ** -48
        assert np.abs(b.get_state(i) - m.rk4(x0, dt, steps)).max() <= steps * np.abs(x0).max() * eps
    b.destroy()
    for s in systems:
        s.destroy()


def test_success_leaves_the_error_text():
    """qh_last_error() is the message of the last failure, not of steps that ran"""
    qs, _, _ = build_system(_tc(2, 9))
    A, x0 = qs.matrix(), _start(36)
    v = qa.DeviceVec(len(x0), qa.FP64)
    v.set(x0)
    assert qa.lib().qh_mat_set_lanes(A.h, 3, 0) != 0
    text = qa.lib().qh_last_error()
    assert b"lanes" in text
    qa.rk4_prepare(A, v, 0.01)
    qa.rk4_device(A, v, 0.01, 3)
    assert qa.lib().qh_last_error() == text
    qs.destroy()


@pytest.mark.parametrize("recipe", [_tc(2, 12), _noisy(5, [("ham", 0.3 + 0.1 * i, [(i, "sx")]) for i in range(5)])],
                         ids=["closed sets", "stage kernels"])
def test_renormalised_every_odd_number_of_steps(recipe):
    """the trace is one after exactly renorm_every steps, and the steps after it leave it"""
    qs, _, _ = build_system(recipe)
    A, n = qs.matrix(), qs.total_levels
    x0 = 1.5 * _start(n)
    for every, steps in ((5, 5), (3, 9), (1, 4), (7, 16)):
        f = _steps(A, x0, qa.FP32, 0.01, steps, tot=n, renorm_every=every)
        # the two words' rounding of n entries, and of a step that keeps the trace
        assert abs(np.trace(f.reshape(n, n)) - 1.0) < 1e-12 + (steps % every) * n * 2.0 ** -24, (every, steps)
    f = _steps(A, x0, qa.FP32, 0.01, 4, tot=n, renorm_every=5)
    assert abs(np.trace(f.reshape(n, n)) - 1.5) < 4 * n * 2.0 ** -24
    qs.destroy()


@pytest.mark.parametrize("prec", [qa.FP64, qa.FP32])
@pytest.mark.parametrize("recipe", [_noisy(8), _noisy(9)], ids=["8", "9"])
def test_short_calls_step_the_same_state(recipe, prec):
    """one step a call (all bins in one launch) and many (a launch a shape, some on the
    side stream) are the same arithmetic"""
    qs, _, _ = build_system(recipe)
    A, n, dt, steps = qs.matrix(), qs.total_levels, 0.02, 200
    x0 = _start(n)
    one = _steps(A, x0, prec, dt, steps)
    v = qa.DeviceVec(len(x0), prec)
    v.set(x0)
    for _ in range(steps):
        qa.rk4_device(A, v, dt, 1)
    # FP64: bitwise; FP32: the state is split into its two words between the calls
    assert np.abs(v.get() - one).max() <= (0.0 if prec == qa.FP64 else steps * np.abs(x0).max() * 2.0 ** -48)
    tot, terms = recipes.oracle_terms(recipe)
    ref = oracle.construct(tot, terms, dm=True).rk4(x0, dt, 5)
    rp, _, val = A.export()
    norm = np.add.reduceat(np.abs(val), rp[:-1]).max()
    tol = 5 * np.abs(x0).max() * (2 * dt * norm + 8) * (2.0 ** -53 if prec == qa.FP64 else 2.0 ** -47)
    assert np.abs(_steps(A, x0, prec, dt, 5) - ref).max() <= tol + (2.0 ** -47 if prec == qa.FP32 else 0.0)
    qs.destroy()


@pytest.mark.parametrize("prec", [qa.FP64, qa.FP32])
def test_plan_is_formed_when_it_pays(prec):
    """a few FP64 steps run without a plan and without a choice of variant; the plan
    follows when as many steps have run, and the state goes on from where it is; an FP32
    state has its plan, which steps it in 64 bits, at once"""
    recipe, dt = _tc(2, 13), 0.02
    qs, _, _ = build_system(recipe)
    A, n = qs.matrix(), qs.total_levels
    x0 = _start(n)
    tot, terms = recipes.oracle_terms(recipe)
    m = oracle.construct(tot, terms, dm=True)
    rp, _, val = A.export()
    norm = np.add.reduceat(np.abs(val), rp[:-1]).max()
    v = qa.DeviceVec(len(x0), prec)
    v.set(x0)
    formed = 0
    for k in range(1, 41):
        qa.rk4_device(A, v, dt, 1)
        if not formed and A.closed_info(prec)["bins"]:
            formed = k
        if k in (1, 3, 40):
            # a few roundings of the state and of h A times it a step
            eps = 2.0 ** -53 if prec == qa.FP64 else 2.0 ** -47
            assert np.abs(v.get() - m.rk4(x0, dt, k)).max() <= (k + 1) * np.abs(x0).max() * (2 * dt * norm + 8) * eps, k
    assert (3 <= formed <= 20 if prec == qa.FP64 else formed == 1) and A.lanes() == (0, 0)
    B, _, _ = build_system(recipe)
    v.set(x0)
    qa.rk4_device(B.matrix(), v, dt, 40)  # enough steps in one call
    assert B.matrix().closed_info(prec)["bins"] > 0
    for s in (qs, B):
        s.destroy()


def test_refused_plan_is_looked_at_once():
    """one set of 4096 rows: the stage kernels step it, the second matrix of the size
    without another look"""
    recipe = _noisy(6, [("ham", 0.3 + 0.1 * i, [(i, "sx")]) for i in range(6)])
    x0, dt = _start(64), 0.01
    tot, terms = recipes.oracle_terms(recipe)
    m = oracle.construct(tot, terms, dm=True)
    for steps in (60, 3):
        qs, _, _ = build_system(recipe)
        v = qa.DeviceVec(len(x0), qa.FP64)
        v.set(x0)
        qa.rk4_device(qs.matrix(), v, dt, steps)
        assert qs.matrix().closed_info()["bins"] == 0 and qs.matrix().lanes()[0] != 0
        rp, _, val = qs.matrix().export()
        norm = np.add.reduceat(np.abs(val), rp[:-1]).max()
        tol = steps * np.abs(x0).max() * (2 * dt * norm + 8) * 2.0 ** -53
        assert np.abs(v.get() - m.rk4(x0, dt, steps)).max() <= tol
        qs.destroy()

"""Time-dependent terms whose entries A's uniform slots take over (variant 134, FP64):
all of them, some (a drive on an operator that A does not hold, or with values that
differ within a slot), none, and more dictionary entries than the kernel holds,
against the CSR kernel in both integrators."""
import math

import numpy as np
import pytest

import quac_amd as qa
from qbuild import build_system

pytestmark = pytest.mark.gpu


def _chain(dims):
    terms = []
    for s, n in enumerate(dims):
        terms.append(("ham", 0.5 + 0.1 * s, [(s, "sx")]) if n == 2 else ("ham", 0.2, [(s, "n")]))
        terms.append(("lin", 0.03, [(s, "lower")]))
    return {"subs": [("op", n) for n in dims], "terms": terms, "mcwf": False}


@pytest.mark.parametrize("method", ["rk4", "rk3bs"])
@pytest.mark.parametrize("dims,drives", [
    ((2,) * 5, [(0, "sx"), (1, "sx"), (4, "sx")]),             # every entry
    ((2,) * 5, [(0, "sx"), (1, "sy"), (2, "sz")]),             # the first only
    ((2, 2, 2, 5), [(0, "sx"), (3, "lower"), (3, "raise")]),   # a cavity's entries stay
    ((2,) * 5, [(0, "sz")]),                                   # nothing
    ((2, 2, 9), [(0, "sx"), (2, "n"), (2, "lower"), (2, "raise")]),
    ((2,) * 5, [(k % 5, "sx") for k in range(33)]),            # two dictionary entries a term: too many
])
def test_folded_drives(dims, drives, method):
    out = []
    for lanes in (8, 134):
        qs, _, op = build_system(_chain(dims), construct=False)
        for k, ref in enumerate(drives):
            qs.add_ham_term_time_dep(0.3 / (1 + k), lambda t, k=k: math.cos((1 + 0.3 * k) * t), op(ref))
        qs.construct_matrix()
        qs.matrix().set_lanes(lanes, 0)
        qa.set_option("ts_rk_type", "4" if method == "rk4" else "3bs")
        qa.set_option("ts_adapt_type", "none" if method == "rk4" else "basic")
        n = int(np.prod(dims))
        rng = np.random.default_rng(7)
        psi = rng.normal(size=n) + 1j * rng.normal(size=n)
        x = qs.create_qvec()
        x.set(np.outer(psi.conj(), psi).reshape(-1) / np.linalg.norm(psi) ** 2)
        steps, _ = qs.time_step(x, 0.0, 0.3, 0.01, 10 ** 6)
        out.append((steps, x.get()))
        x.destroy()
        qs.destroy()
    qa.set_option("ts_rk_type", "4")
    qa.set_option("ts_adapt_type", "none")
    assert out[0][0] == out[1][0]
    # roundings in another order, a few a step (h A is below 1), and of the step sizes
    assert np.abs(out[0][1] - out[1][1]).max() <= out[0][0] * 64 * np.abs(out[0][1]).max() * 2.0 ** -53

"""Performance cases: the work that programs on this library have it do, through
its Python API (quac_amd), over the range of sizes they meet.

Every case is an open quantum system: build it (prepare), then one pass (run) of
what the program repeats -- integrate a state for a stretch of time, step a batch
of a parameter sweep, alternate gates and noise, advance Monte Carlo trajectories,
solve for a steady state, or take one new parameter set from its terms to its
result.  Parameters and initial states come from the seed.

    listed()            the cases
    draw(rng)           one more case of the same ranges
    prepare(case, seed) the state of a program before the pass
    run(state)          one pass; its outputs
    work(case)          bytes and flops a pass cannot do without
    tolerance(case)     how far another correct implementation may be off
    exact(case, seed)   the outputs of run in 64 bits by plain torch
"""
import ctypes
import math
import random

import numpy as np
import torch

import quac_amd as qa

# ------------------------------------------------------------------ the cases
# system: jc (two-level emitter and a cavity of `levels`), tc (`qubits` emitters
# and a cavity of `levels`), chain (`qubits` in a dissipative Ising chain), noisy
# (`qubits` with decay and dephasing only), kerr (three driven cavities of
# `levels`).
# do: evolve (one state, fixed RK4 steps or the default adaptive integrator),
# sweep (a batch of tc systems), circuit (layers of gates with noise between),
# mcwf (trajectories), steady (a new set of terms to its steady state), fresh (a
# new set of terms to its populations).


def listed():
    return [
        # the textbook system, integrated between two read-outs: 400 superoperator
        # rows, so that latency counts
        {"name": "jc_rk4", "do": "evolve", "system": "jc", "levels": 10, "method": "rk4", "bits": 64, "steps": 100},
        # the same system with the integrator that a program gets without options
        {"name": "jc_adaptive", "do": "evolve", "system": "jc", "levels": 10, "method": "rk3bs", "bits": 64,
         "time": 20.0},
        # one member of a sweep run by itself: 18 496 rows, four launches a step
        {"name": "tc_rk4", "do": "evolve", "system": "tc", "qubits": 3, "levels": 17, "method": "rk4", "bits": 64,
         "steps": 100},
        # one new parameter set from its terms to its populations, an odd cavity
        {"name": "tc_fresh", "do": "fresh", "system": "tc", "qubits": 2, "levels": 23, "steps": 50},
        # a parameter sweep of uneven sizes in one batch: 100 to 230 400 rows each
        {"name": "tc_sweep", "do": "sweep", "instances": 512, "steps": 20, "renorm": 10},
        # the spin chain, rho 1024 x 1024, in both precisions
        {"name": "chain10_rk4", "do": "evolve", "system": "chain", "qubits": 10, "method": "rk4", "bits": 64,
         "steps": 40},
        {"name": "chain10_rk4_fp32", "do": "evolve", "system": "chain", "qubits": 10, "method": "rk4", "bits": 32,
         "steps": 40},
        # and with the default integrator
        {"name": "chain10_adaptive", "do": "evolve", "system": "chain", "qubits": 10, "method": "rk3bs", "bits": 64,
         "time": 0.5},
        # the chain under three time-dependent drives
        {"name": "chain10_driven", "do": "evolve", "system": "chain", "qubits": 10, "method": "rk4", "bits": 64,
         "steps": 20, "drives": 3},
        # gates and noise in turn on a 4096 x 4096 density matrix
        {"name": "circuit12", "do": "circuit", "system": "noisy", "qubits": 12, "layers": 2, "gates": 8, "steps": 10},
        # an ensemble of Monte Carlo trajectories, every jump located
        {"name": "jc_mcwf", "do": "mcwf", "system": "jc", "levels": 10, "trajectories": 10000, "steps": 500},
        # one parameter set of the driven cavities to its steady state
        {"name": "kerr_steady", "do": "steady", "system": "kerr", "levels": 8},
    ]


def _log(rng, lo, hi):
    """an integer spread over the logarithm of [lo, hi]"""
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    do = rng.choice(["evolve", "evolve", "evolve", "evolve", "sweep", "circuit", "mcwf", "steady", "fresh"])
    if do == "sweep":
        return {"do": do, "instances": _log(rng, 8, 512), "steps": rng.randint(5, 20), "renorm": rng.choice([0, 5, 10])}
    if do == "circuit":
        return {"do": do, "system": "noisy", "qubits": rng.randint(5, 12), "layers": rng.randint(1, 2),
                "gates": rng.randint(2, 8), "steps": rng.randint(3, 10)}
    if do == "mcwf":
        return {"do": do, "system": "jc", "levels": rng.randint(3, 24), "trajectories": _log(rng, 200, 10000),
                "steps": rng.randint(50, 500)}
    if do == "steady":
        return {"do": do, "system": "kerr", "levels": rng.randint(3, 8)}
    if do == "fresh":
        return {"do": do, "system": "tc", "qubits": rng.randint(1, 4), "levels": rng.randint(5, 30),
                "steps": rng.randint(10, 60)}
    system = rng.choice(["jc", "tc", "chain"])
    c = {"do": do, "system": system, "method": rng.choice(["rk4", "rk4", "rk3bs"])}
    if system == "chain":
        c["qubits"] = rng.randint(4, 10)
    elif system == "tc":
        c["qubits"], c["levels"] = rng.randint(1, 4), rng.randint(5, 30)
    else:
        c["levels"] = rng.randint(3, 24)
    c["bits"] = 64 if c["method"] == "rk3bs" else rng.choice([64, 32])
    if c["method"] == "rk4":
        c["steps"] = rng.randint(5, 40) if system == "chain" else rng.randint(20, 150)
        if rng.random() < 0.25:
            c["drives"] = rng.randint(1, 3)
    else:
        c["time"] = rng.uniform(0.3, 0.5) if system == "chain" else rng.uniform(1.0, 20.0)
    return c


# ---------------------------------------------------------------- the systems
# A system is its subsystems' levels and its terms: ("ham" | "lin", coefficient,
# [(subsystem, operator), ...]) with the operators lower, raise, n, sx, sz.


def _tc(qubits, levels, rng):
    g, delta = rng.uniform(0.05, 0.2), rng.uniform(-0.1, 0.1)
    kappa, gamma = rng.uniform(1e-3, 1e-2), rng.uniform(1e-3, 1e-2)
    c = qubits
    terms = [("ham", delta, [(c, "n")])]
    for i in range(qubits):
        terms += [("ham", g, [(i, "raise"), (c, "lower")]), ("ham", g, [(c, "raise"), (i, "lower")])]
    terms += [("lin", kappa, [(c, "lower")])] + [("lin", gamma, [(i, "lower")]) for i in range(qubits)]
    return [2] * qubits + [levels], terms


def _system(case, rng):
    kind = case["system"]
    if kind == "tc":
        return _tc(case["qubits"], case["levels"], rng)
    if kind == "jc":
        w, wc, g = rng.uniform(0.8, 1.2), rng.uniform(0.8, 1.2), rng.uniform(0.05, 0.2)
        return [2, case["levels"]], [
            ("ham", w, [(0, "n")]), ("ham", wc, [(1, "n")]), ("ham", g, [(0, "raise"), (1, "lower")]),
            ("ham", g, [(1, "raise"), (0, "lower")]), ("lin", rng.uniform(5e-3, 2e-2), [(0, "lower")]),
            ("lin", rng.uniform(5e-3, 2e-2), [(1, "lower")])]
    if kind == "kerr":
        kap, hop, terms = rng.uniform(0.05, 0.2), rng.uniform(0.1, 0.5), []
        for k in range(3):
            drive = rng.uniform(0.0, 1.0)
            terms += [("ham", rng.uniform(-1, 1), [(k, "n")]),
                      ("ham", rng.uniform(0.05, 0.5), [(k, "raise"), (k, "raise"), (k, "lower"), (k, "lower")]),
                      ("ham", drive, [(k, "lower")]), ("ham", drive, [(k, "raise")]), ("lin", kap, [(k, "lower")])]
        for k in range(2):
            terms += [("ham", hop, [(k, "raise"), (k + 1, "lower")]), ("ham", hop, [(k + 1, "raise"), (k, "lower")])]
        return [case["levels"]] * 3, terms
    n = case["qubits"]
    if kind == "noisy":
        terms = [("lin", rng.uniform(5e-4, 2e-3), [(i, "lower")]) for i in range(n)]
        return [2] * n, terms + [("lin", rng.uniform(1e-3, 4e-3), [(i, "sz")]) for i in range(n)]
    terms = [("ham", rng.uniform(0.5, 1.5), [(i, "sx")]) for i in range(n)]
    terms += [("ham", rng.uniform(0.5, 1.5), [(i, "sz"), (i + 1, "sz")]) for i in range(n - 1)]
    terms += [("lin", 1e-3, [(i, "lower")]) for i in range(n)] + [("lin", 5e-3, [(i, "sz")]) for i in range(n)]
    return [2] * n, terms


def _drives(case, levels, rng):
    """(coefficient, envelope, operator) of the time-dependent terms: a drive on the
    first subsystems, a quadrature where they have more than two levels"""
    out = []
    for k in range(case.get("drives", 0)):
        w, p = rng.uniform(0.8, 2.0), rng.uniform(0.0, 6.28)
        sub = k % len(levels)
        names = ["sx"] if levels[sub] == 2 else ["lower", "raise"]
        out += [(0.2, (lambda t, w=w, p=p: math.cos(w * t + p)), (sub, name)) for name in names]
    return out


def _psi(levels, rng):
    """a product state: every qubit somewhere on its sphere, every cavity in a
    coherent state of about one photon"""
    psi = np.ones(1, np.complex128)
    for n in levels:
        if n == 2:
            th, ph = rng.uniform(0.0, math.pi), rng.uniform(0.0, 6.28)
            v = np.array([math.cos(th / 2), math.sin(th / 2) * np.exp(1j * ph)])
        else:
            a = rng.uniform(0.5, 1.2) * np.exp(1j * rng.uniform(0.0, 6.28))
            v = np.array([a ** k / math.sqrt(math.factorial(k)) for k in range(n)])
        psi = np.kron(psi, v / np.linalg.norm(v))
    return psi


def _build(levels, terms):
    qs = qa.System()
    ops = [qs.create_op(n) for n in levels]
    pick = {"lower": lambda o: o, "raise": lambda o: o.dag, "n": lambda o: o.n, "sx": lambda o: o.sig_x,
            "sz": lambda o: o.sig_z}
    for kind, a, names in terms:
        add = qs.add_ham_term if kind == "ham" else qs.add_lin_term
        add(a, *[pick[name](ops[sub]) for sub, name in names])
    return qs, ops, pick


def _strides(levels):
    tot = int(np.prod(levels))
    out, before = [], 1
    for n in levels:
        before *= n
        out.append(tot // before)
    return out


class _View:
    """the entries of a device vector, for torch to alias; a tensor made from it
    keeps it, and with it the owner of the vector"""

    def __init__(self, vec, owner):
        f = qa.lib().qh_vec_data
        f.restype, f.argtypes = ctypes.c_void_p, [ctypes.c_void_p]
        self.vec, self.owner = vec, owner
        self.__cuda_array_interface__ = {"shape": (vec.n,), "typestr": "<c16", "data": (f(vec.h), False), "version": 2}


def _tensor(vec, owner):
    view = _View(vec, owner)
    t = torch.as_tensor(view, device="cuda")
    t.view_of = view
    return t


# ------------------------------------------------------------------ a program


def _options(case):
    rk4 = case.get("method", "rk4") == "rk4"
    bits = case.get("bits", 64)
    qa.set_option("ts_rk_type", "4" if rk4 else "3bs")
    qa.set_option("ts_adapt_type", "none" if rk4 else "basic")
    qa.set_option("quac_precision", "fp%d" % bits)
    qa.set_option("quac_renorm", "10" if bits == 32 else "0")


def _dt(case):
    return 0.005 if case.get("system") == "chain" else 0.01


def _gates(case, rng):
    """layers of (name, qubits, angle), every qubit at most once in a layer"""
    layers = []
    for _ in range(case["layers"]):
        qubits, layer = list(range(case["qubits"])), []
        rng.shuffle(qubits)
        while len(layer) < case["gates"] and len(qubits) >= 2:
            name = rng.choice(["H", "CNOT", "RX", "RZ"])
            q = [qubits.pop() for _ in range(2 if name == "CNOT" else 1)]
            layer.append((name, q, rng.uniform(0.0, 6.28) if name[0] == "R" else 0.0))
        layers.append(layer)
    return layers


class _Held:
    """the library's objects that a program holds; they are destroyed with it"""

    def __init__(self):
        self.systems, self.vectors, self.layers, self.batch = [], [], [], None

    def __del__(self):
        for v in self.vectors:
            v.destroy()
        if self.batch is not None:
            self.batch.destroy()
        for c in self.layers:
            c.destroy()
        for qs in self.systems:
            qs.destroy()


def _sweep_parameters(case, rng):
    return [(rng.randint(1, 4), rng.randint(5, 30)) for _ in range(case["instances"])]


def prepare(case, seed):
    # the sizes of a sweep belong to the case, so that its work does not depend on the seed
    rng = random.Random(seed)
    _options(case)
    s = _Held()
    s.case = case
    if case["do"] == "sweep":
        mats, tots, s.subs, blocks = [], [], [], []
        for qubits, levels in _sweep_parameters(case, random.Random(2)):
            dims, terms = _tc(qubits, levels, rng)
            qs, _, _ = _build(dims, terms)
            qs.construct_matrix()
            s.systems.append(qs)
            mats.append(qs.matrix())
            tots.append(int(np.prod(dims)))
            s.subs.append(list(zip(dims, _strides(dims))))
            psi = torch.from_numpy(_psi(dims, rng)).cuda()
            blocks.append(torch.outer(psi.conj(), psi).reshape(-1))
        s.batch = qa.Batch(mats, tots, prec=qa.FP32)
        s.x0 = qa.DeviceVec(sum(n * n for n in tots), qa.FP64)
        s.x = qa.DeviceVec(s.x0.n, qa.FP64)
        _tensor(s.x0, s).copy_(torch.cat(blocks))
        torch.cuda.synchronize()
        return s
    dims, terms = _system(case, rng)
    s.dims = dims
    if case["do"] in ("fresh", "steady"):
        s.terms = terms
        s.psi = _psi(dims, rng)
        return s
    qs, s.ops, pick = _build(dims, terms)
    s.systems.append(qs)
    if case["do"] == "mcwf":
        qs.use_mcwf_solver(case["trajectories"], seed + 1)
        qs.construct_matrix()
        s.psi = _psi(dims, rng)
        return s
    for a, f, (sub, name) in _drives(case, dims, rng):
        qs.add_ham_term_time_dep(a, f, pick[name](s.ops[sub]))
    qs.construct_matrix()
    psi = torch.from_numpy(_psi(dims, rng)).cuda()
    s.x0, s.x = qs.create_qvec(), qs.create_qvec()
    s.vectors += [s.x0, s.x]
    qa.synchronize()
    _tensor(s.x0.data(), s).copy_(torch.outer(psi.conj(), psi).reshape(-1))
    torch.cuda.synchronize()
    if case["do"] == "circuit":
        for layer in _gates(case, rng):
            c = qa.Circuit(len(layer))
            for name, q, theta in layer:
                c.add_gate(1.0, name, q, theta=theta)
            s.layers.append(c)
    return s


def _numbers(x, ops):
    return np.array([x.expectation(o.n).real for o in ops])


def run(s):
    case = s.case
    _options(case)
    if case["do"] == "sweep":
        qa._qh(qa.lib().qh_vec_copy(s.x0.h, s.batch.state().h))
        s.batch.rk4(0.01, case["steps"], renorm_every=case["renorm"])
        pops = s.batch.populations(s.subs)
        qa._qh(qa.lib().qh_vec_copy(s.batch.state().h, s.x.h))
        qa.synchronize()
        return {"state": _tensor(s.x, s), "populations": np.concatenate(pops)}
    if case["do"] in ("fresh", "steady"):
        new = _Held()  # goes with the outputs
        qs, ops, _ = _build(s.dims, s.terms)
        new.systems.append(qs)
        qs.construct_matrix()
        x = qs.create_qvec()
        new.vectors.append(x)
        if case["do"] == "steady":
            qs.steady_state(x, restart=100, tol=1e-10, maxit=2000)
        else:
            x.set(np.outer(s.psi.conj(), s.psi))
            qs.time_step(x, 0.0, 0.01 * case["steps"], 0.01, 10 ** 7)
        return {"populations": _numbers(x, ops), "state": _tensor(x.data(), new)}
    qs = s.systems[0]
    if case["do"] == "mcwf":
        x = qs.create_qvec()
        x.set(s.psi)
        qs.time_step(x, 0.0, 0.01 * case["steps"], 0.01, 10 ** 7)
        out = {"populations": _numbers(x, s.ops), "probabilities": x.bitstring_probs()}
        x.destroy()
        return out
    x = s.x
    qa.lib().copy_qvec(s.x0.h, x.h)
    if case["do"] == "circuit":
        for k, layer in enumerate(s.layers):
            qs.apply_circuit_to_qvec(layer, x)
            qs.time_step(x, 0.01 * k * case["steps"], 0.01 * (k + 1) * case["steps"], 0.01, 10 ** 7)
    else:
        end = case["time"] if case["method"] == "rk3bs" else _dt(case) * case["steps"]
        qs.time_step(x, 0.0, end, _dt(case), 10 ** 7)
    return {"populations": _numbers(x, s.ops), "state": _tensor(x.data(), s)}


# ------------------------------------------------------------------ its bounds


def _entries(dims, terms):
    """entries of a row of the superoperator: the diagonal, two for every
    off-diagonal Hamiltonian term's share of the rows, one for a jump"""
    n = 1.0
    for kind, _, ops in terms:
        if any(name in ("lower", "raise", "sx") for _, name in ops):
            n += 2.0 if kind == "ham" else 0.8
    return n


def _step_work(rows, entries, size):
    """a fourth-order step: four products of the generator with a vector, each
    reading its input and writing its result, and eight flops an entry"""
    return 4 * 2 * size * rows, 4 * 8 * entries * rows


def work(case):
    rng = random.Random(0)
    if case["do"] == "sweep":
        total = [0.0, 0.0]
        for qubits, levels in _sweep_parameters(case, random.Random(2)):
            dims, terms = _tc(qubits, levels, rng)
            b, f = _step_work(int(np.prod(dims)) ** 2, _entries(dims, terms), 8)
            total = [total[0] + b * case["steps"], total[1] + f * case["steps"]]
        return {"bytes": total[0], "flops": total[1]}
    dims, terms = _system(case, rng)
    n, e = int(np.prod(dims)), _entries(dims, terms)
    if case["do"] == "mcwf":
        # amplitudes in and out once; the steps of a trajectory need no memory
        e = 1.0 + (e - 1.0) / 2
        return {"bytes": 32.0 * n * case["trajectories"], "flops": 32.0 * e * n * case["trajectories"] * case["steps"]}
    e += 2.0 * case.get("drives", 0)
    if case["do"] == "steady":
        # about 36 iterations, each four N x N products for the preconditioner, the
        # generator's product, and the basis read twice
        its = 36
        return {"bytes": its * 16.0 * n * n * (its + 4), "flops": its * (16.0 * n ** 3 + 8.0 * e * n * n)}
    if case.get("method") == "rk3bs":
        # the accepted steps of the integrator (about 0.04 each at these tolerances), three products each
        b, f = _step_work(n * n, e, 16)
        steps = max(1.0, case["time"] / (0.04 if case["system"] == "chain" else 0.1)) * 0.75
        return {"bytes": b * steps, "flops": f * steps}
    b, f = _step_work(n * n, e, 16 if case.get("bits", 64) == 64 else 8)
    steps = case["steps"] * case.get("layers", 1)
    if case["do"] == "circuit":
        return {"bytes": b * steps + 32.0 * n * n * case["layers"] * case["gates"], "flops": f * steps}
    return {"bytes": b * steps, "flops": f * steps}


def tolerance(case):
    # measured against exact(), which sums in another order: 32-bit products 2e-9
    # to 2e-8, a solve to a residual of 1e-10 9e-10, fixed steps 1e-16 to 9e-16,
    # adaptive ones (whose step sizes carry the rounding of the error norm) up to
    # 1e-14, trajectories 1e-13
    if case["do"] == "sweep" or case.get("bits") == 32:
        return {"rel": 1e-7, "max": 1e-5}
    if case["do"] == "steady":
        return {"rel": 1e-8, "max": 1e-6}
    if case["do"] == "mcwf" or case.get("method") == "rk3bs":
        return {"rel": 1e-12, "max": 1e-10}
    return {"rel": 1e-14, "max": 1e-11}


# ------------------------------------------------------------ in plain 64 bits
# A density matrix R (row i, column j at entry N j + i of the library's vectors)
# under L(R) = G R + R G^dag + D o R + sum_k a_k C_k R C_k^dag, where
# G = -i H - 1/2 sum_k a_k C_k^dag C_k and D gathers the diagonal jumps.


def _matrix(dims, ops):
    """the product of the operators as (source, value): row r of the result is
    value[r] times row source[r] of what it is applied to"""
    strides = _strides(dims)
    n = int(np.prod(dims))
    src, val = np.arange(n), np.ones(n)
    for sub, name in ops:
        level = (src // strides[sub]) % dims[sub]
        if name == "n":
            val = val * level
        elif name == "sz":
            val = val * (1.0 - 2.0 * level)
        elif name == "sx":
            src = src + np.where(level == 0, 1, -1) * strides[sub]
        elif name == "lower":
            ok = level < dims[sub] - 1
            val, src = np.where(ok, val * np.sqrt(level + 1.0), 0.0), np.where(ok, src + strides[sub], src)
        else:
            ok = level > 0
            val, src = np.where(ok, val * np.sqrt(1.0 * level), 0.0), np.where(ok, src - strides[sub], src)
    return src, val


def _dense(dims, ops):
    src, val = _matrix(dims, ops)
    m = np.zeros((len(src), len(src)))
    m[np.arange(len(src)), src] = val
    return m


class _Generator:
    def __init__(self, dims, terms):
        n = int(np.prod(dims))
        diag = torch.zeros(n, dtype=torch.complex128, device="cuda")
        self.D = torch.zeros(n, n, dtype=torch.complex128, device="cuda")
        off, self.jumps = [], []
        for kind, a, ops in terms:
            src, val = (torch.from_numpy(v).cuda() for v in _matrix(dims, ops))
            own = bool((src == torch.arange(n, device="cuda")).all())
            if kind == "ham":
                if own:
                    diag += -1j * a * val
                else:
                    off.append((-1j * a, src, val))
                continue
            # C^dag C is diagonal: entry src[r] gets value[r]^2
            diag += torch.zeros(n, dtype=torch.float64, device="cuda").index_add_(0, src, val * val) * (-0.5 * a)
            if own:
                self.D += a * torch.outer(val, val)
            else:
                self.jumps.append((src, a * torch.outer(val, val)))
        self.G = None
        if off:
            self.G = torch.diag(diag)
            for c, src, val in off:
                self.G[torch.arange(n, device="cuda"), src] += c * val
            self.Gd = self.G.conj().T.contiguous()
        else:
            self.D += diag[:, None] + diag.conj()[None, :]

    def __call__(self, R):
        out = self.D * R
        if self.G is not None:
            out += self.G @ R
            out += R @ self.Gd
        for src, w in self.jumps:
            out += w * R[src][:, src]
        return out


def _rk4(f, R, t, h):
    k1 = f(t, R)
    k2 = f(t + h / 2, R + h / 2 * k1)
    k3 = f(t + h / 2, R + h / 2 * k2)
    k4 = f(t + h, R + h * k3)
    return R + h / 6 * (k1 + 2 * k2 + 2 * k3 + k4)


def _rk3bs(f, R, t0, t1, h):
    """Bogacki-Shampine 3(2), absolute and relative tolerance 5e-7, next step 0.9
    err^(-1/3) times the last (a factor between 0.1 and 10), kept in [0.01, 1]"""
    t, k1, eps = t0, None, 1e-12 * (abs(t1) + abs(h) + 1.0)
    while t < t1 - eps:
        hh = min(h, t1 - t)
        k1 = f(t, R) if k1 is None else k1
        k2 = f(t + hh / 2, R + hh / 2 * k1)
        k3 = f(t + 3 * hh / 4, R + 3 * hh / 4 * k2)
        new = R + hh * (2 / 9 * k1 + 1 / 3 * k2 + 4 / 9 * k3)
        k4 = f(t + hh, new)
        e = hh * ((2 / 9 - 7 / 24) * k1 + (1 / 3 - 1 / 4) * k2 + (4 / 9 - 1 / 3) * k3 - 1 / 8 * k4)
        scale = 5e-7 + 5e-7 * torch.maximum(R.abs(), new.abs())
        err = float(((e.abs() / scale) ** 2).mean().sqrt())
        h = min(1.0, max(0.01, hh * min(10.0, max(0.1, 0.9 * max(err, 1e-300) ** (-1 / 3)))))
        if err <= 1.0 or hh <= 0.01 * (1 + 1e-12):
            R, k1, t = new, k4, t + hh
    return R


def _populations(R, dims):
    d = torch.diagonal(R).real
    at = torch.arange(len(d), device=d.device)
    return np.array([float((((at // s) % n) * d).sum()) for n, s in zip(dims, _strides(dims))])


def _vector(R):
    return R.T.contiguous().reshape(-1)


def _start(psi):
    psi = torch.from_numpy(psi).cuda()
    return torch.outer(psi, psi.conj())


def _gate(R, dims, name, qubits, theta):
    if name == "H":
        u = np.array([[1, 1], [1, -1]]) / math.sqrt(2)
    elif name == "RX":
        u = np.array([[math.cos(theta / 2), -1j * math.sin(theta / 2)], [-1j * math.sin(theta / 2), math.cos(theta / 2)]])
    elif name == "RZ":
        u = np.diag([1, np.exp(1j * theta)])
    else:
        u = np.array([[1, 0, 0, 0], [0, 1, 0, 0], [0, 0, 0, 1], [0, 0, 1, 0]])
    u = torch.from_numpy(u.astype(np.complex128)).cuda()
    n, k = len(dims), len(qubits)
    for side in (0, 1):  # on the rows, then conjugated on the columns
        axes = [side * n + q for q in qubits]
        T = R.reshape(list(dims) * 2)
        T = torch.tensordot((u if side == 0 else u.conj()).reshape([2] * (2 * k)), T, dims=(list(range(k, 2 * k)), axes))
        R = torch.movedim(T, list(range(k)), axes).reshape(R.shape)
    return R.contiguous()


class _Uniforms:
    """uniforms in [0, 1): xoshiro256** seeded through SplitMix64"""

    MASK = (1 << 64) - 1

    def __init__(self, seed):
        self.s, z = [], seed
        for _ in range(4):
            z = (z + 0x9E3779B97F4A7C15) & self.MASK
            t = ((z ^ (z >> 30)) * 0xBF58476D1CE4E5B9) & self.MASK
            t = ((t ^ (t >> 27)) * 0x94D049BB133111EB) & self.MASK
            self.s.append(t ^ (t >> 31))

    def __call__(self):
        q, m = self.s, self.MASK
        r = (q[1] * 5) & m
        r = (((r << 7) | (r >> 57)) & m) * 9 & m
        t = (q[1] << 17) & m
        q[2] ^= q[0]
        q[3] ^= q[1]
        q[1] ^= q[2]
        q[0] ^= q[3]
        q[2] ^= t
        q[3] = ((q[3] << 45) | (q[3] >> 19)) & m
        return (r >> 11) * 2.0 ** -53


def _trajectories(case, dims, terms, psi, seed):
    """the ensemble: a trajectory jumps where its squared norm reaches its
    threshold, located inside the step; the draws of a round of jumps (operator,
    next threshold) are made in the order of the trajectories"""
    uniform, M, J, h = _Uniforms(seed + 1), case["trajectories"], case["steps"], 0.01
    G = torch.from_numpy(sum((-1j * a * _dense(dims, ops) if kind == "ham" else
                              -0.5 * a * _dense(dims, ops).T @ _dense(dims, ops)) for kind, a, ops in terms)).cuda()
    C = [(a, torch.from_numpy(_dense(dims, ops).astype(np.complex128)).cuda()) for kind, a, ops in terms if kind == "lin"]
    GT = G.T.contiguous()
    X = torch.from_numpy(psi).cuda()[None, :].repeat(M, 1)
    r = torch.tensor([uniform() for _ in range(M)], dtype=torch.float64).cuda()
    j, sub = torch.zeros(M, dtype=torch.int64).cuda(), torch.zeros(M, dtype=torch.float64).cuda()

    def powers(V):
        out = [V]
        for k in range(1, 5):
            out.append(out[-1] @ GT / k)
        return out

    def at(P, t):
        v = P[4]
        for k in (3, 2, 1, 0):
            v = v * t[:, None] + P[k]
        return v

    while True:
        idx = torch.nonzero(j < J).reshape(-1)
        jumped = []
        V, jj, ss, rr = X[idx], j[idx], sub[idx], r[idx]
        while len(idx):
            P = powers(V)
            left = h - ss
            new = at(P, left)
            hit = (new.abs() ** 2).sum(1) < rr
            step = ~hit
            if bool(hit.any()):
                Q = [p[hit] for p in P]
                lo, hi = torch.zeros_like(left[hit]), left[hit].clone()
                for _ in range(60):
                    mid = (lo + hi) / 2
                    above = (at(Q, mid).abs() ** 2).sum(1) > rr[hit]
                    lo, hi = torch.where(above, mid, lo), torch.where(above, hi, mid)
                X[idx[hit]], j[idx[hit]], sub[idx[hit]] = at(Q, hi), jj[hit], ss[hit] + hi
                jumped.append(idx[hit])
            V, jj, ss = torch.where(hit[:, None], V, new), jj + 1, torch.zeros_like(ss)
            done = step & (jj >= J)
            if bool(done.any()):
                X[idx[done]], j[idx[done]], sub[idx[done]] = V[done], jj[done], 0.0
            go = step & (jj < J)
            if not bool(go.all()):
                idx, V, jj, ss, rr = idx[go], V[go], jj[go], ss[go], rr[go]
        if not jumped:
            break
        who = torch.cat(jumped).sort().values
        after = [X[who] @ c.T for _, c in C]
        p = np.array([[a * x for x in (v.abs() ** 2).sum(1).tolist()] for (a, _), v in zip(C, after)]).T
        for q, i in enumerate(who.tolist()):
            tot = p[q].sum()
            if tot > 0.0:
                u, acc, k = uniform(), 0.0, len(C) - 1
                for m in range(len(C)):
                    acc += p[q][m] / tot
                    if acc >= u:
                        k = m
                        break
                X[i] = math.sqrt(C[k][0]) / math.sqrt(p[q][k]) * after[k][q]
            r[i] = uniform()
    prob = X.abs() ** 2
    prob = (prob / prob.sum(1, keepdim=True)).mean(0)
    level = torch.arange(len(prob)).cuda()
    pops = np.array([float((((level // s) % n) * prob).sum()) for n, s in zip(dims, _strides(dims))])
    return {"populations": pops, "probabilities": prob.cpu().numpy()}


def _steady(dims, terms):
    """GMRES on (L + e0 tr) R = e0, preconditioned with the inverse of R -> G R +
    R G^dag in G's eigenbasis"""
    L = _Generator(dims, terms)
    n = L.G.shape[0]
    w, V = np.linalg.eig(L.G.cpu().numpy())
    Vi = torch.from_numpy(np.linalg.inv(V)).cuda()
    w, V = torch.from_numpy(w).cuda(), torch.from_numpy(V).cuda()
    den = w[:, None] + w.conj()[None, :]
    Vh, Vih = V.conj().T.contiguous(), Vi.conj().T.contiguous()

    def pre(R):
        return V @ ((Vi @ R @ Vih) / den) @ Vh

    def op(R):
        out = L(R)
        out[0, 0] += torch.diagonal(R).sum()
        return out

    x = torch.zeros(n, n, dtype=torch.complex128, device="cuda")
    b = x.clone()
    b[0, 0] = 1.0
    for _ in range(20):
        res = b - op(x)
        beta = float(res.abs().square().sum().sqrt())
        if beta < 1e-13:
            break
        Q, H = [(res / beta).reshape(-1)], np.zeros((121, 120), np.complex128)
        for k in range(120):
            v = op(pre(Q[k].reshape(n, n))).reshape(-1)
            B = torch.stack(Q)
            for _ in range(2):
                c = B.conj() @ v
                v = v - c @ B
                H[:k + 1, k] += c.cpu().numpy()
            norm = float(v.abs().square().sum().sqrt())
            H[k + 1, k] = norm
            Q.append(v / norm)
            e = np.zeros(k + 2, np.complex128)
            e[0] = beta
            y, *_ = np.linalg.lstsq(H[:k + 2, :k + 1], e, rcond=None)
            if np.linalg.norm(e - H[:k + 2, :k + 1] @ y) < 2e-14:
                break
        x = x + pre((torch.from_numpy(y).cuda() @ torch.stack(Q[:len(y)])).reshape(n, n))
    return x


def exact(case, seed):
    rng = random.Random(seed)
    if case["do"] == "sweep":
        states, pops = [], []
        for qubits, levels in _sweep_parameters(case, random.Random(2)):
            dims, terms = _tc(qubits, levels, rng)
            R, L = _start(_psi(dims, rng)), _Generator(dims, terms)
            for k in range(case["steps"]):
                R = _rk4(lambda t, R: L(R), R, 0.0, 0.01)
                if case["renorm"] and (k + 1) % case["renorm"] == 0:
                    R = R / torch.diagonal(R).sum().real
            states.append(_vector(R))
            pops.append(_populations(R, dims))
        return {"state": torch.cat(states), "populations": np.concatenate(pops)}
    dims, terms = _system(case, rng)
    if case["do"] == "mcwf":
        return _trajectories(case, dims, terms, _psi(dims, rng), seed)
    if case["do"] == "steady":
        R = _steady(dims, terms)
        return {"populations": _populations(R, dims), "state": _vector(R)}
    L = _Generator(dims, terms)
    drives = [(a, f, torch.from_numpy(_dense(dims, [op]).astype(np.complex128)).cuda())
              for a, f, op in _drives(case, dims, rng)]
    R = _start(_psi(dims, rng))

    def f(t, R):
        out = L(R)
        for a, env, m in drives:
            out += (-1j * a * env(t)) * (m @ R - R @ m)
        return out

    if case["do"] == "circuit":
        for layer in _gates(case, rng):
            for name, q, theta in layer:
                R = _gate(R, dims, name, q, theta)
            for _ in range(case["steps"]):
                R = _rk4(f, R, 0.0, 0.01)
    elif case.get("method") == "rk3bs":
        R = _rk3bs(f, R, 0.0, case["time"], _dt(case))
    else:
        h = _dt(case)
        for k in range(case["steps"]):
            R = _rk4(f, R, k * h, h)
            if case.get("bits", 64) == 32 and (k + 1) % 10 == 0:
                R = R / torch.diagonal(R).sum().real
    return {"populations": _populations(R, dims), "state": _vector(R)}

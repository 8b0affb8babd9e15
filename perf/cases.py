"""Timed cases of the engine: what a user's program calls, over the sizes it is used at.

Kinds of case
  apply      State.apply of a packed op list on |0..0> (or on a given state for
             the QFT): simulate() of a circuit that was not compiled
  compiled   State.apply_schedule of a Schedule made beforehand (mode "auto"):
             simulate() after compile()
  batch      Batch.run: many small variational states, <sum Z> of each
  serve      Server.submit / wait of a burst of mixed requests, states kept
  measure    reductions and sampled shots of a state that is not changed
  collapse   measure_qubit on a few qubits of a copy of a state

Circuits: "brickwork" (U3 on every qubit, CZ on alternating pairs), "random"
(H, X, RZ or RY per qubit, CX on a random matching), "ansatz" (RY and RZ on
every qubit, CX ladder), "qft" (with its final swaps) and "iqft".

States come back as views of their device buffers.  Values that are computed
from a complex64 state and handed over as doubles are returned in 32 bits,
which is what they are good for.  The served indices are not returned: a shot
whose uniform falls between two roundings of the cumulative distribution is
another index, and both are right ("measure" compares indices, on one given
state).
"""
import ctypes
import math

import numpy as np
import torch

from afquantumsim_amd import hip

# ---- circuits ----------------------------------------------------------------
# A gate is (form, target, control, m): "m" 2x2 matrix on the target, "d" the
# diagonal of one, "p" phase m where target (and control) are 1, "x" flip of
# the target, "s" exchange of target and control.  control is None where there
# is none.  Angles are the float32 values that the reference's gates hold.


def _cs(a):
    h = float(np.float32(a)) / 2.0
    return math.cos(h), math.sin(h)


def _h():
    return np.array([1, 1, 1, -1], dtype=np.complex128) * math.sqrt(0.5)


def _ry(a):
    c, s = _cs(a)
    return np.array([c, -s, s, c], dtype=np.complex128)


def _rz(a):
    c, s = _cs(a)
    return np.array([complex(c, -s), 0, 0, complex(c, s)])


def _u3(t, p, l):
    c, s = _cs(t)
    p, l = float(np.float32(p)), float(np.float32(l))
    e = lambda x: complex(math.cos(x), math.sin(x))  # noqa: E731
    return np.array([c, -e(l) * s, e(p) * s, e(p + l) * c])


def _brickwork(n, depth, rng):
    out = []
    for layer in range(depth):
        for q in range(n):
            out.append(("m", q, None, _u3(*rng.uniform(0.0, 2.0 * math.pi, size=3))))
        for a in range(layer % 2, n - 1, 2):
            out.append(("p", a + 1, a, -1.0))
    return out


def _random(n, depth, rng):
    out = []
    for _ in range(depth):
        for q in range(n):
            c, t = int(rng.integers(4)), float(rng.uniform(0.0, 2.0 * math.pi))
            out.append((("m", q, None, _h()), ("x", q, None, None), ("d", q, None, _rz(t)), ("m", q, None, _ry(t)))[c])
        perm = rng.permutation(n)
        for k in range(n // 2):
            out.append(("x", int(perm[2 * k + 1]), int(perm[2 * k]), None))
    return out


def _ansatz(n, depth, rng):
    out = []
    for _ in range(depth):
        out += [("m", q, None, _ry(rng.uniform(-math.pi, math.pi))) for q in range(n)]
        out += [("d", q, None, _rz(rng.uniform(-math.pi, math.pi))) for q in range(n)]
        out += [("x", q + 1, q, None) for q in range(n - 1)]
    return out


def _cphase(i, j, sign):
    a = sign * float(np.float32(math.pi) / np.float32(1 << (i - j)))
    return ("p", i, j, complex(math.cos(a), math.sin(a)))


def _qft(n, depth, rng):
    out = []
    for i in range(n - 1, -1, -1):
        out.append(("m", i, None, _h()))
        out += [_cphase(i, j, 1.0) for j in range(i)]
    return out + [("s", i, n - 1 - i, None) for i in range(n // 2)]


def _iqft(n, depth, rng):
    out = []
    for i in range(n):
        out += [_cphase(i, j, -1.0) for j in range(i - 1, -1, -1)]
        out.append(("m", i, None, _h()))
    return out


_CIRCUITS = {"brickwork": _brickwork, "random": _random, "ansatz": _ansatz, "qft": _qft, "iqft": _iqft}


def _gates(case, seed):
    return _CIRCUITS[case["circuit"]](case["n"], case["depth"], np.random.default_rng(seed))


def _gate_count(circuit, n, depth):
    """(one-qubit matrices, real ones among them, diagonals, two-qubit phases, flips and swaps)."""
    if circuit == "brickwork":
        return n * depth, 0, 0, (n - 1) * depth // 2, 0
    if circuit == "random":
        return n * depth // 2, n * depth // 2, n * depth // 4, 0, n * depth // 4 + n // 2 * depth
    if circuit == "ansatz":
        return n * depth, n * depth, n * depth, 0, (n - 1) * depth
    return n, n, 0, n * (n - 1) // 2, (n // 2 if circuit == "qft" else 0)


def _lower(gates):
    """Gates as the op dicts of the C ABI."""
    out = []
    for form, t, c, m in gates:
        ctl = () if c is None else (c,)
        if form == "m":
            out.append({"kind": hip.OP_MAT1, "targets": (t,), "controls": ctl, "m": m})
        elif form == "d":
            out.append({"kind": hip.OP_DIAG1, "targets": (t,), "controls": ctl, "m": m})
        elif form == "p":
            out.append({"kind": hip.OP_PHASE, "targets": (t,), "controls": ctl, "m": np.array([m, 0, 0, 0], dtype=np.complex128)})
        elif form == "x":
            out.append({"kind": hip.OP_X, "targets": (t,), "controls": ctl})
        else:
            out.append({"kind": hip.OP_SWAP, "targets": (t, c)})
    return out


# ---- cases -------------------------------------------------------------------

_PREC = {"c64": hip.C64, "c128": hip.C128}


def listed():
    return [
        # the reference's own benchmark circuit, at its own size: launches and latency
        {"name": "apply qft 10q", "kind": "apply", "circuit": "qft", "n": 10, "depth": 0, "precision": "c64"},
        # the largest state that one workgroup holds, a circuit of some hundred gates
        {"name": "apply random 12q", "kind": "apply", "circuit": "random", "n": 12, "depth": 30, "precision": "c64"},
        # one state of a variational loop: a short circuit on a medium state
        {"name": "apply ansatz 15q", "kind": "apply", "circuit": "ansatz", "n": 15, "depth": 6, "precision": "c64"},
        # the 20-qubit random circuit of 1200 gates, not compiled
        {"name": "apply random 20q", "kind": "apply", "circuit": "random", "n": 20, "depth": 40, "precision": "c64"},
        # the headline workload's state, some layers of it, gate by gate
        {"name": "apply brickwork 28q", "kind": "apply", "circuit": "brickwork", "n": 28, "depth": 4, "precision": "c64"},
        # the FP64 reference run against which results are checked
        {"name": "apply brickwork 25q c128", "kind": "apply", "circuit": "brickwork", "n": 25, "depth": 3, "precision": "c128"},
        # compile() below the cache sizes: a served request's circuit
        {"name": "compiled random 17q", "kind": "compiled", "circuit": "random", "n": 17, "depth": 40, "precision": "c64"},
        # compile() of the headline workload
        {"name": "compiled brickwork 28q", "kind": "compiled", "circuit": "brickwork", "n": 28, "depth": 20, "precision": "c64"},
        # compile() of the largest QFT
        {"name": "compiled qft 30q", "kind": "compiled", "circuit": "qft", "n": 30, "depth": 0, "precision": "c64"},
        # a variational sweep: states of 10..16 qubits, 4..12 layers
        {"name": "batch ansatz 512", "kind": "batch", "count": 512, "nmin": 10, "nmax": 16, "lmin": 4, "lmax": 12},
        # a burst of small and medium requests
        {"name": "serve brickwork 24", "kind": "serve", "count": 24, "nmin": 12, "nmax": 18, "lmin": 10, "lmax": 40, "shots": 1000},
        # profile_measure_all and the expectation values of a large state
        {"name": "measure 27q", "kind": "measure", "n": 27, "precision": "c64", "shots": 1000},
    ]


# amplitudes times gates of the largest listed case of a kind
_MOST = {"apply": 160 << 28, "compiled": 800 << 28}


def draw(rng):
    kind = rng.choice(["apply", "apply", "apply", "compiled", "compiled", "compiled", "batch", "serve", "measure", "collapse"])
    if kind in ("apply", "compiled"):
        circuit = rng.choice(["brickwork", "brickwork", "random", "random", "ansatz", "ansatz", "qft", "iqft"])
        precision = rng.choice(["c64", "c64", "c64", "c128"])
        n = rng.randint(6, 28 if kind == "apply" else 29)
        if precision == "c128":
            n = min(n, 24 + rng.randint(0, 2))
        depth = 0
        if circuit not in ("qft", "iqft"):
            depth = int(round(math.exp(rng.uniform(math.log(3), math.log(60)))))
        most = _MOST[kind] >> (2 if precision == "c128" else 0)
        while sum(_gate_count(circuit, n, depth)) << n > most:
            if depth > 2:
                depth -= 1
            else:
                n -= 1
        return {"kind": kind, "circuit": circuit, "n": n, "depth": depth, "precision": precision}
    if kind == "batch":
        nmin = rng.randint(4, 12)
        lmin = rng.randint(2, 6)
        return {"kind": "batch", "count": int(round(math.exp(rng.uniform(math.log(17), math.log(480))))), "nmin": nmin,
                "nmax": min(16, nmin + rng.randint(1, 6)), "lmin": lmin, "lmax": lmin + rng.randint(0, 6)}
    if kind == "serve":
        nmin = rng.randint(8, 15)
        lmin = rng.randint(5, 20)
        return {"kind": "serve", "count": rng.randint(3, 24), "nmin": nmin, "nmax": min(18, nmin + rng.randint(0, 5)),
                "lmin": lmin, "lmax": lmin + rng.randint(0, 20), "shots": rng.randint(10, 1000)}
    precision = rng.choice(["c64", "c64", "c128"])
    n = rng.randint(8, 27 if precision == "c64" else 26)
    if kind == "measure":
        return {"kind": "measure", "n": n, "precision": precision, "shots": int(round(math.exp(rng.uniform(math.log(7), math.log(20000)))))}
    return {"kind": "collapse", "n": n, "precision": precision, "qubits": rng.randint(1, 3)}


# ---- states ------------------------------------------------------------------


class _Buffer:
    """A state's device buffer under the array interface."""

    def __init__(self, state):
        p = ctypes.c_void_p()
        hip.check(hip.load().aqs_state_device_ptr(state.h, ctypes.byref(p)))
        self.state = state
        self.__cuda_array_interface__ = {"shape": (1 << state.n,), "typestr": "<c8" if state.precision == hip.C64 else "<c16",
                                         "data": (p.value, False), "version": 2}


def _view(state):
    return torch.as_tensor(_Buffer(state), device="cuda")


def _input(n, precision, seed):
    """A random state of norm 1 on the device."""
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed))
    real = torch.float32 if precision == "c64" else torch.float64
    x = torch.randn((1 << n, 2), generator=g, dtype=real, device="cuda")
    x /= torch.linalg.vector_norm(x.view(-1), dtype=torch.float64).to(real)
    return torch.view_as_complex(x)


def _given_state(n, precision, seed):
    st = hip.State(n, _PREC[precision])
    _view(st).copy_(_input(n, precision, seed))
    torch.cuda.synchronize()
    return st


def _circuit_case(case, seed):
    packed = hip.PackedOps(_lower(_gates(case, seed)))
    st = hip.State(case["n"], _PREC[case["precision"]])
    given = _given_state(case["n"], case["precision"], seed) if case["circuit"] in ("qft", "iqft") else None
    return {"kind": case["kind"], "state": st, "view": _view(st), "given": given, "ops": packed}


def _members(case):
    """(qubits, layers) of a batch's states or a burst's requests: the case's own, angles come from the seed."""
    rng = np.random.default_rng([case["count"], case["nmin"], case["nmax"], case["lmin"], case["lmax"]])
    return [(int(rng.integers(case["nmin"], case["nmax"] + 1)), int(rng.integers(case["lmin"], case["lmax"] + 1)))
            for _ in range(case["count"])]


def prepare(case, seed):
    kind = case["kind"]
    hip.init(0)
    if kind == "apply":
        return _circuit_case(case, seed)
    if kind == "compiled":
        s = _circuit_case(case, seed)
        s["schedule"] = hip.Schedule(s["ops"], case["n"], mode="auto")
        return s
    if kind == "batch":
        rng = np.random.default_rng(seed)
        return {"kind": kind, "batch": hip.Batch([(n, _lower(_ansatz(n, depth, rng))) for n, depth in _members(case)])}
    if kind == "serve":
        rng = np.random.default_rng(seed)
        reqs = [(n, hip.PackedOps(_lower(_brickwork(n, depth, rng))), rng.uniform(size=case["shots"]))
                for n, depth in _members(case)]
        return {"kind": kind, "server": hip.Server(16 << 30, workers=4), "requests": reqs, "next": 0}
    rng = np.random.default_rng(seed)
    given = _given_state(case["n"], case["precision"], seed)
    if kind == "measure":
        return {"kind": kind, "state": given, "u": rng.uniform(size=case["shots"])}
    st = hip.State(case["n"], _PREC[case["precision"]])
    qubits = [int(q) for q in rng.permutation(case["n"])[: case["qubits"]]]
    # uniforms that are not within rounding of a random state's P(1) = 1/2
    return {"kind": kind, "state": st, "view": _view(st), "given": given, "qubits": qubits,
            "u": [float(rng.uniform(0.0, 0.3) + 0.7 * rng.integers(2)) for _ in qubits]}


def run(s):
    kind = s["kind"]
    if kind in ("apply", "compiled"):
        st = s["state"]
        if s["given"] is not None:
            st.copy_from(s["given"])
        else:
            st.set_basis(0)
        if kind == "apply":
            st.apply(s["ops"])
        else:
            st.apply_schedule(s["schedule"])
        return s["view"]
    if kind == "batch":
        z, _ = s["batch"].run()
        return z.astype(np.float32)
    if kind == "serve":
        srv, first = s["server"], s["next"]
        s["next"] += len(s["requests"])
        for k, (n, ops, u) in enumerate(s["requests"]):
            srv.submit(first + k, n, ops, u, keep_state=True)
        return [srv.wait(first + k)[2] for k in range(len(s["requests"]))]
    if kind == "measure":
        st = s["state"]
        return {"p1": st.prob1_all(), "z": st.expect_sum_z(), "shots": st.sample(s["u"]).astype(np.int64)}
    st = s["state"]
    st.copy_from(s["given"])
    got = [st.measure_qubit(q, u) for q, u in zip(s["qubits"], s["u"])]
    return {"state": s["view"], "outcomes": [o for o, _ in got], "p1": np.array([p for _, p in got], dtype=np.float32)}


# ---- work --------------------------------------------------------------------


def _circuit_flops(circuit, n, depth):
    mats, real, diag, phases, _ = _gate_count(circuit, n, depth)
    per_amp = 14.0 * (mats - real) + 6.0 * real + 6.0 * diag + 6.0 * 0.25 * phases
    return per_amp * (1 << n)


def work(case):
    kind = case["kind"]
    if kind in ("apply", "compiled"):
        state = (8 if case["precision"] == "c64" else 16) << case["n"]
        given = case["circuit"] in ("qft", "iqft")
        return {"bytes": state * (2 if given else 1), "flops": _circuit_flops(case["circuit"], case["n"], case["depth"])}
    if kind in ("batch", "serve"):
        circuit = "ansatz" if kind == "batch" else "brickwork"
        ns = range(case["nmin"], case["nmax"] + 1)
        depth = (case["lmin"] + case["lmax"]) // 2
        mean = lambda f: sum(f(n) for n in ns) / len(ns)  # noqa: E731
        return {"bytes": case["count"] * mean(lambda n: 8.0 * (1 << n)),
                "flops": case["count"] * mean(lambda n: _circuit_flops(circuit, n, depth))}
    state = (8 if case["precision"] == "c64" else 16) << case["n"]
    if kind == "measure":
        # |a|^2 once, its sum for every qubit and the cumulative sum
        return {"bytes": state, "flops": (4.0 + case["n"]) * (1 << case["n"])}
    return {"bytes": 2 * state, "flops": 4.0 * (1 << case["n"])}


# ---- the same in 64 bits ---------------------------------------------------------


def _part(psi, n, fixed):
    """The view of psi with index bits fixed ({qubit: value})."""
    shape, index, run_len = [], [], 1
    for q in range(n):
        if q in fixed:
            if run_len > 1:
                shape.append(run_len)
                index.append(slice(None))
            shape.append(2)
            index.append(fixed[q])
            run_len = 1
        else:
            run_len *= 2
    shape.append(run_len)
    index.append(slice(None))
    return psi.view(shape)[tuple(index)]


def _run_exact(psi, n, gates):
    for form, t, c, m in gates:
        ctl = {} if c is None else {c: 1}
        if form == "p":
            _part(psi, n, {t: 1, **ctl}).mul_(complex(m))
        elif form == "s":
            a, b = _part(psi, n, {t: 1, c: 0}), _part(psi, n, {t: 0, c: 1})
            keep = a.clone()
            a.copy_(b)
            b.copy_(keep)
        else:
            a, b = _part(psi, n, {t: 0, **ctl}), _part(psi, n, {t: 1, **ctl})
            if form == "x":
                keep = a.clone()
                a.copy_(b)
                b.copy_(keep)
            elif form == "d":
                a.mul_(complex(m[0]))
                b.mul_(complex(m[3]))
            else:
                na = a * complex(m[0])
                na.add_(b, alpha=complex(m[1]))
                nb = b * complex(m[3])
                nb.add_(a, alpha=complex(m[2]))
                a.copy_(na)
                b.copy_(nb)
    return psi


def _zero_state(n, count=1):
    psi = torch.zeros(count << n, dtype=torch.complex128, device="cuda")
    psi[:: 1 << n] = 1
    return psi


def _batch_exact(case, seed):
    """States of the same size and depth together: every gate has one target for all and a matrix for each."""
    rng = np.random.default_rng(seed)
    groups = {}
    for i, (n, depth) in enumerate(_members(case)):
        groups.setdefault((n, depth), []).append((i, _ansatz(n, depth, rng)))
    z = torch.zeros(case["count"], dtype=torch.float64, device="cuda")
    for (n, _), members in groups.items():
        k = len(members)
        psi = _zero_state(n, k).view(k, -1)
        mats = np.array([[g[3] if g[3] is not None else np.zeros(4) for g in gates] for _, gates in members])
        mats = torch.from_numpy(mats).to("cuda")
        for j, (form, t, c, _) in enumerate(members[0][1]):
            if form == "x":
                v = psi.view(k, 1 << c, 2, 2, -1)  # the ladder's control is the qubit before its target
                v[:, :, 1] = v[:, :, 1].flip(2)
                continue
            v = psi.view(k, 1 << t, 2, -1)
            m = mats[:, j].view(k, 4, 1, 1)
            a, b = v[:, :, 0], v[:, :, 1]
            if form == "d":
                a.mul_(m[:, 0])
                b.mul_(m[:, 3])
            else:
                na, nb = m[:, 0] * a + m[:, 1] * b, m[:, 2] * a + m[:, 3] * b
                a.copy_(na)
                b.copy_(nb)
        p = psi.real.square() + psi.imag.square()
        index = torch.arange(1 << n, device="cuda")
        ones = sum((index >> q) & 1 for q in range(n))
        z[[i for i, _ in members]] = p @ (n - 2 * ones).double()
    return z


def exact(case, seed):
    kind = case["kind"]
    if kind in ("apply", "compiled"):
        n = case["n"]
        psi = _input(n, case["precision"], seed).to(torch.complex128) if case["circuit"] in ("qft", "iqft") else _zero_state(n)
        return _run_exact(psi, n, _gates(case, seed))
    if kind == "batch":
        return _batch_exact(case, seed)
    if kind == "serve":
        rng = np.random.default_rng(seed)
        out = []
        for n, depth in _members(case):
            out.append(_run_exact(_zero_state(n), n, _brickwork(n, depth, rng)))
            rng.uniform(size=case["shots"])
        # laid out as the host arrays that the server hands over
        return [x.cpu().numpy() for x in out]
    psi = _input(case["n"], case["precision"], seed).to(torch.complex128)
    n = case["n"]
    p = psi.real.square() + psi.imag.square()
    if kind == "measure":
        p1 = [_part(p, n, {q: 1}).sum() for q in range(n)]
        total = p.sum()
        return {"p1": torch.stack(p1).cpu().numpy(), "z": float(sum(total - 2 * x for x in p1)), "shots": None}
    rng = np.random.default_rng(seed)
    qubits = [int(q) for q in rng.permutation(n)[: case["qubits"]]]
    us = [float(rng.uniform(0.0, 0.3) + 0.7 * rng.integers(2)) for _ in qubits]
    seen = []
    for q, u in zip(qubits, us):
        ones = psi.real.square() + psi.imag.square()
        p1 = float(_part(ones, n, {q: 1}).sum())
        one = u < p1
        kept = p1 if one else float(_part(ones, n, {q: 0}).sum())
        _part(psi, n, {q: 0 if one else 1}).zero_()
        psi *= 1.0 / math.sqrt(kept)
        seen.append(p1)
    return {"state": psi, "outcomes": None, "p1": np.array(seen)}

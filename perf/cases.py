"""The engine's work as its users call it, for timing and comparison.

Every case goes through the package's public calls and returns what such a
call is made for: amplitudes, <Z> and <ZZ> values, Pauli expectation values,
sampled outcomes or counts. Values of single-precision states are handed on in
single precision (the ABI widens them to double).

A case is a dict of plain values; its "kind" names the path:

  run          run(circuit, shots) of a few qubits with a measurement and
               feedback in the middle: the call a notebook or a test makes
  statevector  statevector(circuit) of a random circuit over the whole gate set
  estimator    expectation(circuit, observable): one evaluation of a
               variational circuit with fresh angles
  circuit      set_zero, apply_ops and expectation values on a state that is kept: the
               random benchmark circuit on a product state, a Trotterised
               kicked-Ising circuit, or the QFT of a product state
  fused        the same for a circuit fused to dense gates of up to `width`
               qubits, each applied in its own pass (no tiles)
  steps        a program that applies its gates one call at a time (dense,
               controlled and diagonal) and measures and resets on the way
               (these three end with <Z>, <ZZ> and two strings of X and Y)
  sample       outcomes for given uniforms from a dense state that is kept
  batch        one evaluation of many small variational circuits
"""
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))),
                                "qevedo-simulator_amd", "python"))

from qevedo.simulator import Batch, Circuit, StateVector, expectation, library, lower_gates, run as run_circuit  # noqa: E402
from qevedo.simulator import _native, statevector  # noqa: E402


def listed():
    return [
        # The smallest call: a five-qubit program with a mid-circuit
        # measurement, where latency and launches count.
        {"name": "run_5q", "kind": "run", "qubits": 5, "gates": 16, "shots": 1000, "precision": "single"},
        # The final state of a small circuit in double precision, as printed
        # or compared in a notebook.
        {"name": "statevector_12q", "kind": "statevector", "qubits": 12, "gates": 120},
        # One evaluation of a variational loop: 6 layers, 40 Pauli terms.
        {"name": "estimator_16q", "kind": "estimator", "qubits": 16, "layers": 6, "terms": 40, "precision": "double"},
        # The random benchmark circuit where the state fits the cache, ...
        {"name": "random_20q", "kind": "circuit", "circuit": "random", "qubits": 20, "depth": 20, "precision": "single"},
        # ... and at the size the benchmark quotes.
        {"name": "random_30q", "kind": "circuit", "circuit": "random", "qubits": 30, "depth": 20, "precision": "single"},
        # Dynamics in double precision: 20 Trotter steps on a heavy-hex patch.
        {"name": "ising_25q_c128", "kind": "circuit", "circuit": "ising", "qubits": 25, "depth": 20, "precision": "double"},
        # The Fourier transform of a product state.
        {"name": "qft_27q", "kind": "circuit", "circuit": "qft", "qubits": 27, "depth": 1, "precision": "single"},
        # Fused dense gates without tiles: 6-qubit gates in single precision
        # and 4-qubit ones (the default width) in double.
        {"name": "fused6_27q", "kind": "fused", "qubits": 27, "depth": 14, "width": 6, "precision": "single"},
        {"name": "fused4_25q_c128", "kind": "fused", "qubits": 25, "depth": 14, "width": 4, "precision": "double"},
        # Gates one call at a time, with measurements between them.
        {"name": "steps_25q", "kind": "steps", "qubits": 25, "rounds": 3, "precision": "single"},
        # 10^6 shots of a dense state.
        {"name": "sample_24q", "kind": "sample", "qubits": 24, "shots": 1000000, "precision": "single"},
        # 256 variational circuits of mixed sizes, <Z> and <ZZ> of each.
        {"name": "batch_256", "kind": "batch", "count": 256, "low": 12, "high": 22, "layers": 6, "precision": "single"},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["run", "statevector", "estimator", "circuit", "circuit", "circuit", "fused", "steps", "sample", "batch"])
    precision = rng.choice(["single", "double"])
    double = precision == "double"
    if kind == "run":
        return {"kind": kind, "qubits": rng.randint(2, 12), "gates": _log_int(rng, 6, 60), "shots": _log_int(rng, 50, 20000),
                "precision": precision}
    if kind == "statevector":
        return {"kind": kind, "qubits": rng.randint(1, 18), "gates": _log_int(rng, 10, 300)}
    if kind == "estimator":
        return {"kind": kind, "qubits": rng.randint(2, 20), "layers": rng.randint(1, 8), "terms": _log_int(rng, 1, 120),
                "precision": "double"}
    if kind == "circuit":
        circuit = rng.choice(["random", "ising", "qft"])
        return {"kind": kind, "circuit": circuit, "qubits": rng.randint(10, 26 if double else 28),
                "depth": 1 if circuit == "qft" else rng.randint(4, 20), "precision": precision}
    if kind == "fused":
        return {"kind": kind, "qubits": rng.randint(12, 25 if double else 27), "depth": rng.randint(4, 14),
                "width": rng.randint(1, 6), "precision": precision}
    if kind == "steps":
        return {"kind": kind, "qubits": rng.randint(3, 25 if double else 26), "rounds": rng.randint(1, 3), "precision": precision}
    if kind == "sample":
        return {"kind": kind, "qubits": rng.randint(8, 23 if double else 24), "shots": _log_int(rng, 100, 1000000),
                "precision": precision}
    low = rng.randint(4, 20)
    return {"kind": kind, "count": _log_int(rng, 2, 200), "low": low, "high": rng.randint(low, 22 if low < 20 else 21),
            "layers": rng.randint(1, 6), "precision": "single"}


# ---------------------------------------------------------------------------
# Inputs.
# ---------------------------------------------------------------------------
def _run_program(case, seed):
    """Instructions of a small program: random gates, a measurement of qubit 0
    with feedback on it, random gates, and a measurement of up to 5 qubits."""
    n = case["qubits"]
    half = case["gates"] // 2
    first = [("gate", g) for g in library.random_gate_circuit(n, half, 2 * seed + 1)]
    second = [("gate", g) for g in library.random_gate_circuit(n, case["gates"] - half, 2 * seed + 2)]
    m = min(n, 4)
    middle = [("measure", (0, m)), ("feedback", ("x", 1, m))]
    return first + middle + second + [("measure", (q, q)) for q in range(m)], m + 1


def _circuit_gates(case, seed):
    n = case["qubits"]
    rng = np.random.default_rng(seed)
    if case["kind"] == "fused" or case["circuit"] == "random":
        return ([("ry", (q,), (float(rng.uniform(0.3, 2.8)),)) for q in range(n)]
                + library.random_circuit(n, case["depth"], seed))
    if case["circuit"] == "ising":
        return library.kicked_ising(n, library.heavy_hex_edges(n), case["depth"], float(rng.uniform(0.1, 1.5)))
    gates = []
    for q in range(n):
        gates.append(("ry", (q,), (float(rng.uniform(0.3, 2.8)),)))
        gates.append(("rz", (q,), (float(rng.uniform(0.0, 6.2)),)))
    return gates + library.qft(n)


def _pauli_labels(n, terms, seed):
    rng = np.random.default_rng(seed + 77)
    labels = {}
    while len(labels) < min(terms, 4 ** n - 1):
        labels.setdefault("".join(rng.choice(list("IXYZ"), n, p=[0.6, 0.13, 0.07, 0.2])), float(rng.normal()))
    return labels


def _transverse(n):
    """X and Z masks of the strings X_0 X_1 ... X_(n-1) and Y_(n/2): values that depend on the phases."""
    return [(1 << n) - 1, 1 << (n // 2)], [0, 1 << (n // 2)]


def _unitary(rng, k):
    m = rng.normal(size=(1 << k, 1 << k)) + 1j * rng.normal(size=(1 << k, 1 << k))
    return np.linalg.qr(m)[0]


def _steps_program(case, seed):
    """("apply", matrix, targets, controls) / ("measure" | "reset", qubit, uniform) in order."""
    rng = np.random.default_rng(seed)
    n = case["qubits"]
    h = np.array([[1, 1], [1, -1]]) / math.sqrt(2)
    steps = [("apply", h, [q], []) for q in range(n)]
    for _ in range(case["rounds"]):
        for k in (1, 2, 2, 3):
            qs = [int(q) for q in rng.permutation(n)[:k + 1]]
            if k <= len(qs) - 1 or n > k:
                steps.append(("apply", _unitary(rng, min(k, n - 1)), qs[:min(k, n - 1)], []))
        qs = [int(q) for q in rng.permutation(n)[:3]]
        steps.append(("apply", np.array([[0, 1], [1, 0]], dtype=complex), qs[:1], [(qs[1], True)]))
        steps.append(("apply", _unitary(rng, 1), qs[:1], [(qs[1], True), (qs[2], False)]))
        steps.append(("apply", np.diag(np.exp(1j * rng.uniform(0, 6.2, 4))), qs[1:3], []))
        steps.append(("measure", int(rng.integers(n)), float(rng.random())))
        steps.append(("reset", int(rng.integers(n)), float(rng.random())))
    return steps


def _batch_sizes(case):
    lo, hi = case["low"], case["high"]
    rng = np.random.default_rng([case["count"], lo, hi])
    sizes = [int(x) for x in rng.integers(lo, hi + 1, size=case["count"])]
    sizes[0] = hi
    return sizes


def _random_amplitudes(n, seed):
    rng = np.random.default_rng(seed)
    v = rng.standard_normal(2 << n, dtype=np.float64)
    v *= 1.0 / math.sqrt(float(v @ v))
    return v.view(np.complex128)


def prepare(case, seed):
    kind = case["kind"]
    if kind == "run":
        instructions, clbits = _run_program(case, seed)
        c = Circuit(case["qubits"], clbits)
        for what, args in instructions:
            if what == "gate":
                c.gate(*args)
            elif what == "measure":
                c.measure(*args)
            else:
                c.feedback(*args)
        return {"case": case, "circuit": c, "seed": seed}
    if kind in ("statevector", "estimator"):
        n = case["qubits"]
        gates = (library.random_gate_circuit(n, case["gates"], seed) if kind == "statevector"
                 else library.hardware_efficient_ansatz(n, case["layers"], seed))
        c = Circuit(n)
        for name, qubits, params in gates:
            c.gate(name, qubits, params)
        return {"case": case, "circuit": c, "observable": _pauli_labels(n, case["terms"], seed) if kind == "estimator" else None}
    if kind in ("circuit", "fused"):
        return {"case": case, "ops": _native.OpArray(lower_gates(_circuit_gates(case, seed))),
                "state": StateVector(case["qubits"], case["precision"])}
    if kind == "steps":
        return {"case": case, "steps": _steps_program(case, seed), "state": StateVector(case["qubits"], case["precision"])}
    if kind == "sample":
        sv = StateVector(case["qubits"], case["precision"])
        sv.set_amplitudes(_random_amplitudes(case["qubits"], seed))
        return {"case": case, "state": sv, "uniforms": np.random.default_rng(seed + 1).random(case["shots"]),
                "out": np.empty(case["shots"], dtype=np.uint64)}
    circuits = [(n, _native.OpArray(lower_gates(library.hardware_efficient_ansatz(n, case["layers"], 1000 * seed + i))))
                for i, n in enumerate(_batch_sizes(case))]
    return {"case": case, "batch": Batch(circuits, case["precision"])}


# ---------------------------------------------------------------------------
# One pass.
# ---------------------------------------------------------------------------
def _typed(case, a):
    return np.asarray(a, dtype=np.float32 if case["precision"] == "single" else np.float64)


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "run":
        r = run_circuit(state["circuit"], case["shots"], seed=state["seed"], precision=case["precision"])
        bits = state["circuit"].num_clbits
        return {"counts": np.array([r.counts.get(format(k, "0%db" % bits), 0) for k in range(1 << bits)], dtype=np.int64)}
    if kind == "statevector":
        return {"amplitudes": statevector(state["circuit"])}
    if kind == "estimator":
        return {"value": _typed(case, [expectation(state["circuit"], state["observable"], precision=case["precision"])])}
    if kind == "sample":
        return {"outcomes": state["state"].sample(state["uniforms"], out=state["out"])}
    if kind == "batch":
        values = state["batch"].run()
        return {"z": _typed(case, np.concatenate([z for z, _ in values])),
                "zz": _typed(case, np.concatenate([zz for _, zz in values]))}
    sv = state["state"]
    sv.set_zero()
    out = {}
    if kind == "steps":
        outcomes = []
        for step in state["steps"]:
            if step[0] == "apply":
                sv.apply(step[1], step[2], step[3])
            elif step[0] == "measure":
                outcomes.append(sv.measure(step[1], step[2]))
            else:
                sv.reset(step[1], step[2])
        out["outcomes"] = np.array(outcomes, dtype=np.int64)
    elif kind == "fused":
        sv.apply_ops(state["ops"], max_fused_qubits=case["width"], tile_bits=None)
    else:
        sv.apply_ops(state["ops"])
    z, zz = sv.expect_z()
    out["z"], out["zz"] = _typed(case, z), _typed(case, zz)
    out["x"] = _typed(case, sv.expect_pauli(*_transverse(case["qubits"])))
    return out


# ---------------------------------------------------------------------------
# Work and 64-bit values.
# ---------------------------------------------------------------------------
def work(case):
    """Bytes: the state written once and read once (for a batch, each state;
    for the applied fused or single gates, one read and one write per pass
    that no fusion of the caller's request removes), and what goes to or
    comes from the host. Flops: 14 per amplitude and dense one-qubit gate (a
    2 x 2 complex matrix), 8 * 2^k per amplitude and dense k-qubit gate, 6 per
    changed amplitude of a phase."""
    kind = case["kind"]
    elem = 16 if case.get("precision", "double") == "double" else 8
    if kind == "batch":
        sizes = _batch_sizes(case)
        amps = float(sum(1 << n for n in sizes))
        gates = sum((1 << n) * n * case["layers"] * 14 for n in sizes)
        return {"bytes": 2 * amps * elem, "flops": float(gates)}
    n = case["qubits"]
    amps = float(1 << n)
    if kind == "run":
        return {"bytes": 2 * amps * elem + 8 * case["shots"], "flops": 14 * amps * case["gates"] + 4 * amps}
    if kind == "statevector":
        return {"bytes": 2 * amps * 16, "flops": 14 * amps * case["gates"]}
    if kind == "estimator":
        return {"bytes": 2 * amps * elem, "flops": amps * (14 * n * case["layers"] + 8 * case["terms"])}
    if kind == "sample":
        return {"bytes": amps * elem + 16 * case["shots"], "flops": 3 * amps}
    if kind == "steps":
        passes = n + 9 * case["rounds"]
        return {"bytes": 2 * amps * elem * passes, "flops": amps * (14 * n + case["rounds"] * 200)}
    gates = _circuit_gates(case, 1)
    one = sum(1 for g in gates if len(g[1]) == 1 and g[0] != "rz")
    two = len(gates) - one
    if kind == "fused":
        w = case["width"]
        passes = max(1, math.ceil(len(gates) / (3.0 * w)))  # about what greedy fusion leaves
        return {"bytes": 2 * amps * elem * passes, "flops": amps * passes * 8 * (1 << w)}
    return {"bytes": 2 * amps * elem, "flops": amps * (14 * one + 1.5 * two)}


def _matrix(name, p):
    """(controls, base matrix) of a gate, Qiskit's conventions."""
    c, s = (math.cos(p[0] / 2), math.sin(p[0] / 2)) if p else (0.0, 0.0)
    e = lambda t: complex(math.cos(t), math.sin(t))  # noqa: E731
    x = [[0, 1], [1, 0]]
    table = {
        "h": lambda: (0, [[math.sqrt(0.5), math.sqrt(0.5)], [math.sqrt(0.5), -math.sqrt(0.5)]]),
        "x": lambda: (0, x), "cx": lambda: (1, x), "ccx": lambda: (2, x),
        "z": lambda: (0, [[1, 0], [0, -1]]), "cz": lambda: (1, [[1, 0], [0, -1]]), "y": lambda: (0, [[0, -1j], [1j, 0]]),
        "rx": lambda: (0, [[c, -1j * s], [-1j * s, c]]), "ry": lambda: (0, [[c, -s], [s, c]]),
        "rz": lambda: (0, [[e(-p[0] / 2), 0], [0, e(p[0] / 2)]]),
        "u3": lambda: (0, [[c, -e(p[2]) * s], [e(p[1]) * s, e(p[1] + p[2]) * c]]),
        "t": lambda: (0, [[1, 0], [0, e(math.pi / 4)]]),
        "sx": lambda: (0, [[0.5 + 0.5j, 0.5 - 0.5j], [0.5 - 0.5j, 0.5 + 0.5j]]),
        "cp": lambda: (1, [[1, 0], [0, e(p[0])]]),
        "rzz": lambda: (0, np.diag([e(-p[0] / 2), e(p[0] / 2), e(p[0] / 2), e(-p[0] / 2)])),
        "swap": lambda: (0, [[1, 0, 0, 0], [0, 0, 1, 0], [0, 1, 0, 0], [0, 0, 0, 1]]),
        "cswap": lambda: (1, [[1, 0, 0, 0], [0, 0, 1, 0], [0, 1, 0, 0], [0, 0, 0, 1]]),
    }
    controls, m = table[name]()
    return controls, np.asarray(m, dtype=complex)


class _State:
    """A state in 64 bits by plain tensor operations. One-qubit matrices are
    collected per qubit until another op needs the qubit."""

    def __init__(self, n, amplitudes=None):
        self.n = n
        device = "cuda" if torch.cuda.is_available() else "cpu"
        if amplitudes is None:
            self.s = torch.zeros(1 << n, dtype=torch.complex128, device=device)
            self.s[0] = 1
        else:
            self.s = torch.as_tensor(amplitudes, dtype=torch.complex128).to(device).clone()
        self.one = {}

    def _apply(self, m, targets, controls):
        order = sorted(list(targets) + [q for q, _ in controls], reverse=True)
        shape, last = [], self.n  # one axis of 2 per qubit of the op, the others merged
        for q in order:
            shape += [1 << (last - q - 1), 2]
            last = q
        v = self.s.view(shape + [1 << last])
        at = [slice(None)] * (2 * len(order) + 1)
        for q, value in controls:
            at[2 * order.index(q) + 1] = int(value)
        parts = []
        for j in range(1 << len(targets)):
            for b, q in enumerate(targets):
                at[2 * order.index(q) + 1] = (j >> b) & 1
            parts.append(v[tuple(at)])
        if not np.count_nonzero(m - np.diag(np.diag(m))):
            for j, part in enumerate(parts):
                if m[j, j] != 1:
                    part.mul_(complex(m[j, j]))
            return
        old = [p.clone() for p in parts]
        for r, part in enumerate(parts):
            first = True
            for k in np.flatnonzero(m[r]):
                if first:
                    torch.mul(old[k], complex(m[r, k]), out=part) if part.is_contiguous() else part.copy_(old[k] * complex(m[r, k]))
                else:
                    part.add_(old[k], alpha=complex(m[r, k]))
                first = False
            if first:
                part.zero_()

    def _flush(self, qubits):
        for q in qubits:
            if q in self.one:
                self._apply(self.one.pop(q), [q], [])

    def op(self, m, targets, controls=()):
        m = np.asarray(m, dtype=complex)
        if len(targets) == 1 and not controls:
            self.one[targets[0]] = m @ self.one.get(targets[0], np.eye(2))
            return
        self._flush(list(targets) + [q for q, _ in controls])
        self._apply(m, list(targets), list(controls))

    def gates(self, gates):
        for name, qubits, params in gates:
            c, m = _matrix(name, params)
            self.op(m, list(qubits[c:]), [(q, 1) for q in qubits[:c]])
        return self

    def amplitudes(self):
        self._flush(list(self.one))
        return self.s

    def _p(self):
        s = self.amplitudes()
        return s.real.square() + s.imag.square()

    def z(self):
        p = self._p()
        z, zz = [], []
        for q in range(self.n):
            t = p.view(-1, 2, 1 << q).sum(dim=(0, 2))
            z.append(float(t[0] - t[1]))
        for q in range(self.n - 1):
            t = p.view(-1, 2, 2, 1 << q).sum(dim=(0, 3))
            zz.append(float(t[0, 0] + t[1, 1] - t[0, 1] - t[1, 0]))
        return np.array(z), np.array(zz)

    def collapse(self, q, uniform):
        p1 = float(self._p().view(-1, 2, 1 << q)[:, 1].sum())
        one = uniform < min(max(p1, 0.0), 1.0)
        v = self.s.view(-1, 2, 1 << q)
        v[:, 0 if one else 1] = 0
        v[:, 1 if one else 0] /= math.sqrt(p1 if one else 1.0 - p1)
        return int(one)

    def pauli(self, label):
        """<P>, Qiskit's label order."""
        s = self.amplitudes()
        i = torch.arange(1 << self.n, device=s.device)
        j = i.clone()
        sign = torch.zeros_like(i)
        phase = 1
        for q, ch in enumerate(reversed(label)):
            bit = (i >> q) & 1
            if ch in "XY":
                j ^= 1 << q
            if ch in "ZY":
                sign ^= bit
            if ch == "Y":
                phase *= 1j  # Y|b> = i (-1)^b |1 - b>
        value = (s[j].conj() * s * (1 - 2 * sign)).sum() * phase
        return float(value.real)


def exact(case, seed):
    kind = case["kind"]
    if kind in ("run", "sample"):
        return None  # whole numbers
    n = case.get("qubits", 0)
    if n > 28:
        return None
    if kind == "statevector":
        s = _State(n).gates(library.random_gate_circuit(n, case["gates"], seed)).amplitudes()
        return {"amplitudes": s.cpu().numpy()}
    if kind == "estimator":
        s = _State(n).gates(library.hardware_efficient_ansatz(n, case["layers"], seed))
        return {"value": np.array([sum(c * s.pauli(p) for p, c in _pauli_labels(n, case["terms"], seed).items())])}
    if kind == "batch":
        values = [_State(m).gates(library.hardware_efficient_ansatz(m, case["layers"], 1000 * seed + i)).z()
                  for i, m in enumerate(_batch_sizes(case))]
        return {"z": np.concatenate([z for z, _ in values]), "zz": np.concatenate([zz for _, zz in values])}
    s = _State(n)
    out = {}
    if kind == "steps":
        for step in _steps_program(case, seed):
            if step[0] == "apply":
                s.op(step[1], step[2], step[3])
            else:
                s.amplitudes()
                one = s.collapse(step[1], step[2])
                if step[0] == "reset" and one:
                    s.op(np.array([[0, 1], [1, 0]]), [step[1]])
        out["outcomes"] = None
    else:
        s.gates(_circuit_gates(case, seed))
    out["z"], out["zz"] = s.z()
    out["x"] = np.array([s.pauli("X" * n), s.pauli("I" * (n - 1 - n // 2) + "Y" + "I" * (n // 2))])
    return out

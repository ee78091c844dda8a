"""Runs of sign and phase pairs over register, thread and non-tile bits (14
qubits: one complex64 tile, no non-tile qubit; 17: three), against the oracle. In
complex64 the engine's bound of 1e-5; FP64 rounding of 300 gates stays under 1e-12."""
import numpy as np
import pytest

from helpers import oracle_statevector, rel_l2
from qevedo.simulator import StateVector, lower_gates

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision,tol", [("single", 1e-5), ("double", 1e-12)])
@pytest.mark.parametrize("n", [14, 17])
@pytest.mark.parametrize("pairs", ["signs", "phases", "both"])
def test_pair_runs(pairs, n, precision, tol):
    r = np.random.default_rng(n)
    gates = [("ry", (q,), (float(r.uniform(0.3, 2.8)),)) for q in range(n)]
    for _ in range(300):
        a, b = (int(q) for q in r.permutation(n)[:2])
        kind = {"signs": ["cz"], "phases": ["cp", "rzz"], "both": ["cz", "cp", "rzz"]}[pairs] + ["h"]
        name = kind[int(r.integers(len(kind)))]
        gates.append((name, (a,) if name == "h" else (a, b), (float(r.uniform(0, 6)),) if name in ("cp", "rzz") else ()))
    with StateVector(n, precision) as sv:
        sv.apply_ops(lower_gates(gates))
        assert rel_l2(sv.amplitudes(), oracle_statevector(n, gates)) < tol

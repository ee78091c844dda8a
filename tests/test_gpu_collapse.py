"""Measurement and reset of states on both sides of the size (27 qubits) from which
qubits inside a 128-byte line take a kernel of their own, against the projector
(and the flip) as ops of the stage kernel on the device. Each side rounds every
amplitude once or twice."""
import numpy as np
import pytest

from qevedo.simulator import StateVector, library, lower_gates

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision,n,qubits", [("single", 26, (0, 3)), ("single", 27, (0, 1, 3, 4)),
                                                ("double", 27, (0, 2, 3))])
@pytest.mark.parametrize("outcome", [0, 1])
@pytest.mark.parametrize("reset", [False, True])
def test_against_the_projector(precision, n, qubits, outcome, reset):
    state = lower_gates(library.random_circuit(n, 2, 7))
    for q in qubits:
        with StateVector(n, precision) as a, StateVector(n, precision) as b:
            a.apply_ops(state)
            b.apply_ops(state)
            p = a.probability_one(q) if outcome else 1 - a.probability_one(q)
            if reset:
                a.reset(q, -1.0 if outcome else 2.0)
            else:
                assert a.measure(q, -1.0 if outcome else 2.0) == outcome
            b.apply_ops([([q], [], np.diag([0, 1 / np.sqrt(p)] if outcome else [1 / np.sqrt(p), 0]).astype(complex))])
            if reset and outcome:
                b.apply_ops(lower_gates([("x", (q,), ())]))
            assert a.compare(b)["rel_l2"] < (3e-7 if precision == "single" else 6e-16)

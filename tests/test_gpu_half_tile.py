"""complex128 stages with two workgroups per CU (22 qubits: 512 tiles, the
fewest that run so), against the oracle in 64 bits: sign and phase runs,
exchanges, the first stages of a fresh state (some of them on few tiles), a
dense state, and a plan whose in-LDS ops keep some stages on the whole-tile
kernel. A gate rounds each amplitude by a few units of 2^-53: 1e-12 covers 600."""
import numpy as np
import pytest

from helpers import oracle_statevector, random_state, rel_l2, rng
from oracle import oracle
from qevedo.simulator import StateVector, library, lower_gates

pytestmark = pytest.mark.gpu


def circuit(kind, n):
    if kind == "random":
        return library.random_circuit(n, 8, 5)
    if kind == "ising":
        return library.kicked_ising(n, library.heavy_hex_edges(n), 3, 0.7)
    if kind == "qft":
        return [("ry", (q,), (0.3 + 0.1 * q,)) for q in range(n)] + library.qft(n)
    return library.random_gate_circuit(n, 120, 9)  # swaps among them


@pytest.mark.parametrize("kind", ["random", "ising", "qft", "gates"])
def test_against_the_oracle(kind):
    n = 22
    gates = circuit(kind, n)
    want = oracle_statevector(n, gates)
    with StateVector(n, "double") as sv:
        sv.apply_ops(lower_gates(gates))
        assert rel_l2(sv.amplitudes(), want) < 1e-12


def test_dense_state():
    n = 22
    gates = circuit("random", n)
    psi = random_state(rng(3), n)
    with oracle.OracleState(n, "double") as o:
        o.set_amplitudes(psi)
        o.apply_ops(oracle.lower(gates), 4, 14)
        want = o.amplitudes()
    with StateVector(n, "double") as sv:
        sv.set_amplitudes(psi)
        sv.apply_ops(lower_gates(gates))
        assert rel_l2(sv.amplitudes(), want) < 1e-12

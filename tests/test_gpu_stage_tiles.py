"""The LDS-tile stage kernel where its split changes: tiles of one wave, four and
sixteen, ops of fewer groups than threads, more ops than one load of records
holds, and the state made in the tile, against the oracle in 64 bits. A
complex128 op rounds each amplitude by at most 18 units of 2^-53 (16 products and
sums): 200 of them stay under 1e-12; complex64 is held to 1e-5, the engine's bound."""
import numpy as np
import pytest

from helpers import oracle_statevector, rel_l2
from qevedo.simulator import StateVector, library, lower_gates

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision,tol", [("single", 1e-5), ("double", 1e-12)])
@pytest.mark.parametrize("width", [1, 4])
@pytest.mark.parametrize("n,tile_bits", [(1, 0), (5, 0), (6, 0), (7, 0), (9, 0), (10, 0), (12, 0), (9, 6), (11, 9), (14, 11)])
def test_tiles_against_the_oracle(n, tile_bits, width, precision, tol):
    gates = library.random_gate_circuit(n, 200, 17 * n + width)
    want = oracle_statevector(n, gates)
    with StateVector(n, precision) as sv:
        for again in range(2):  # the second pass over a state that has to be set anew
            sv.set_zero()
            sv.apply_ops(lower_gates(gates), max_fused_qubits=width, tile_bits=tile_bits)
            assert rel_l2(sv.amplitudes(), want) < tol, again
        sv.set_zero()
        sv.apply_ops(lower_gates(gates[:100]), max_fused_qubits=width, tile_bits=tile_bits)
        sv.apply_ops(lower_gates(gates[100:]), max_fused_qubits=width, tile_bits=tile_bits)
        assert rel_l2(sv.amplitudes(), want) < tol

"""Plans without tiles, whose ops are launched while later ones are still being
fused: more matrices than the arena holds at once, a fresh and a kept state,
and a width that is refused. 400 gates of FP64 rounding stay under 1e-12."""
import pytest

from helpers import oracle_statevector, rel_l2
from qevedo.simulator import NativeError, StateVector, library, lower_gates

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,gates,width", [(9, 12, 1), (9, 400, 2), (10, 400, 6), (8, 6000, 6)])
def test_against_the_oracle(n, gates, width):
    circuit = library.random_gate_circuit(n, gates, 3 * n + width)
    want = oracle_statevector(n, circuit)
    with StateVector(n, "double") as sv:
        sv.apply_ops(lower_gates(circuit), max_fused_qubits=width, tile_bits=None)
        assert rel_l2(sv.amplitudes(), want) < 1e-12
        sv.set_zero()
        st = sv.apply_ops(lower_gates(circuit[: gates // 2]), max_fused_qubits=width, tile_bits=None, timing=True)
        assert st["passes"] == st["kernels"] > 0 and st["other_kernel_seconds"] > 0 and st["stages"] == 0
        sv.apply_ops(lower_gates(circuit[gates // 2:]), max_fused_qubits=width, tile_bits=None)
        assert rel_l2(sv.amplitudes(), want) < 1e-12


def test_too_wide_is_refused():
    with StateVector(9, "single") as sv:
        with pytest.raises(NativeError, match="not supported"):
            sv.apply_ops(lower_gates([("h", (q,), ()) for q in range(9)]), max_fused_qubits=8, tile_bits=None)

"""Plans without tiles on both sides of the state size (16 MiB) from which ops
are launched while later ones are being fused: more matrices than the arena holds
at once, a fresh and a kept state, and a width that is refused, against the tile
plan on the device. 2000 gates of FP64 rounding stay under 1e-12."""
import pytest

from qevedo.simulator import NativeError, StateVector, library, lower_gates

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,gates,width", [(19, 300, 3), (20, 300, 1), (20, 2000, 6), (21, 300, 4)])
def test_against_the_tile_plan(n, gates, width):
    ops = lower_gates(library.random_gate_circuit(n, gates, 3 * n + width))
    with StateVector(n, "double") as a, StateVector(n, "double") as b:
        a.apply_ops(ops, max_fused_qubits=width, tile_bits=None)
        b.apply_ops(ops)
        assert a.compare(b)["rel_l2"] < 1e-12
        a.set_zero()
        st = a.apply_ops(ops[: gates // 2], max_fused_qubits=width, tile_bits=None, timing=True)
        assert st["passes"] == st["kernels"] > 0 and st["other_kernel_seconds"] > 0 and st["stages"] == 0
        a.apply_ops(ops[gates // 2:], max_fused_qubits=width, tile_bits=None)
        assert a.compare(b)["rel_l2"] < 1e-12


def test_too_wide_is_refused():
    with StateVector(21, "single") as sv:
        with pytest.raises(NativeError, match="not supported"):
            sv.apply_ops(lower_gates([("h", (q,), ()) for q in range(9)]), max_fused_qubits=8, tile_bits=None)

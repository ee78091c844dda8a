"""Plans without tiles on both sides of the state size (16 MiB) from which ops
are launched while later ones are being fused: more matrices than the arena holds
at once, a fresh and a kept state, and a width that is refused, against the tile
plan on the device. 2000 gates of FP64 rounding stay under 1e-12."""
import os
import subprocess
import sys

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


MEMORY = """
import numpy as np
from qevedo.simulator import StateVector
from qevedo.simulator._native import OpArray

def status(field):
    with open("/proc/self/status") as f:
        return next(int(l.split()[1]) << 10 for l in f if l.startswith(field))

u = np.linalg.qr(np.random.default_rng(1).normal(size=(64, 64)))[0].astype(complex)
arr = OpArray([([0, 1, 2, 3, 4, 5] if i % 2 else [3, 4, 5, 6, 7, 8], [], u) for i in range(3000)])
with StateVector(20, "double") as sv:
    sv.apply_ops([([0], [], np.eye(2)[::-1])], max_fused_qubits=6, tile_bits=None)
    before = status("VmRSS")
    sv.apply_ops(arr, max_fused_qubits=6, tile_bits=None)
    print(status("VmHWM") - before)
"""


def test_host_copies_are_let_go_on_the_way():
    """3000 gates on 6 qubits that do not fuse: the engine's own ops hold their
    matrices (64 KiB each), the copies on their way to the device no more than the
    4 MiB arena does."""
    out = subprocess.run([sys.executable, "-c", MEMORY], check=True, capture_output=True, text=True, timeout=100,
                         env={**os.environ, "PYTHONPATH": os.pathsep.join(sys.path)}).stdout
    assert int(out) < 1.4 * 3000 * 64 * 1024

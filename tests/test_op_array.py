"""The op array handed to the engine: every form of targets, controls and
matrices it takes reads back as given, and wrong shapes are refused."""
import numpy as np
import pytest

from qevedo.simulator import _native

H = np.array([[1, 1], [1, -1]]) / np.sqrt(2)


def read(arr, i):
    o = arr.arr[i]
    k = 1 << o.num_targets
    return ([o.targets[j] for j in range(o.num_targets)],
            [(o.controls[j], bool(o.control_values[j])) for j in range(o.num_controls)],
            np.array([o.matrix[j] for j in range(2 * k * k)]).view(np.complex128).reshape(k, k))


def test_forms():
    two = np.arange(16).reshape(4, 4) + 1j
    ops = [([3], [], H), ((1, 0), [(5, True), (2, False)], two), (np.array([7, 4], dtype=np.int64), ((6, 1, "x"),), two),
           (2, [], H.tolist()), ([0], [(np.int64(1), 0)], np.asfortranarray(H * 1j)), ([], [], [[1]]),
           ([9, 8], [], two[::-1])]
    arr = _native.OpArray(ops)
    assert arr.n == len(ops)
    for i, (t, c, m) in enumerate(ops):
        targets, controls, matrix = read(arr, i)
        assert targets == [int(q) for q in np.atleast_1d(t)]
        assert controls == [(int(x[0]), bool(x[1])) for x in c]
        assert np.array_equal(matrix, np.asarray(m, dtype=complex))
    assert _native.OpArray([]).n == 0


@pytest.mark.parametrize("targets,matrix", [([0, 1], H), ([0], np.eye(4)), ([0], np.ones(4)), ([], H)])
def test_wrong_shapes_are_refused(targets, matrix):
    with pytest.raises(ValueError, match="needs a"):
        _native.OpArray([([0], [], H), (targets, [], matrix)])


@pytest.mark.parametrize("params", [[0.3], (0.3,), np.array([0.3]), 0.3, np.float64(0.3), ["0.3"]])
def test_gate_parameters(params):
    c, m = _native.gate_lower("rx", params)
    want = np.array([[np.cos(0.15), -1j * np.sin(0.15)], [-1j * np.sin(0.15), np.cos(0.15)]])
    assert c == 0 and np.max(np.abs(m - want)) < 1e-15 and m.flags.writeable

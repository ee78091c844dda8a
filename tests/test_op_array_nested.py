"""Forms of targets, controls and parameters that NumPy flattens: accepted, and read
back as given."""
import numpy as np
import pytest

from qevedo.simulator import _native


@pytest.mark.parametrize("targets", [[[3], [1]], [[3, 1]], ((3, 1),), [np.array([3, 1])], [np.array(3), np.uint8(1)],
                                     np.array([[3], [1]]), [3.0, 1.0], ["3", "1"], [np.int64(3), 1]])
@pytest.mark.parametrize("controls", [[], [(np.array([6]), True)], [(np.int32(6), 1)], np.array([[6, 1]])])
def test_flattened_qubits(targets, controls):
    m = np.arange(16).reshape(4, 4) + 0j
    arr = _native.OpArray([([0], [(2, False)], np.eye(2)), (targets, controls, m), ([5], [], np.eye(2))])
    o = arr.arr[1]
    assert [o.targets[j] for j in range(o.num_targets)] == [3, 1]
    assert [(o.controls[j], o.control_values[j]) for j in range(o.num_controls)] == [(6, 1)] * len(controls)
    assert [o.matrix[j] for j in range(32)] == m.view(float).ravel().tolist()
    assert arr.arr[0].control_values[0] == 0 and arr.arr[2].targets[0] == 5


def test_negative_and_ragged_qubits_are_refused():
    for targets in ([-1, 2], [0, [1]]):
        with pytest.raises((OverflowError, ValueError)):
            _native.OpArray([(targets, [], np.eye(4))])


@pytest.mark.parametrize("params", [[[0.3]], ((0.3,),), [np.array([0.3])], np.array([[0.3]]), [["0.3"]]])
def test_flattened_parameters(params):
    c, m = _native.gate_lower("rx", params)
    assert c == 0 and np.array_equal(m, _native.gate_lower("rx", [0.3])[1])


def test_flattened_parameters_of_several():
    want = _native.gate_lower("u", [0.1, 0.2, 0.3])[1]
    for params in ([[0.1, 0.2, 0.3]], [[0.1], [0.2], [0.3]], [np.array([0.1, 0.2, 0.3])]):
        assert np.array_equal(_native.gate_lower("u", params)[1], want)

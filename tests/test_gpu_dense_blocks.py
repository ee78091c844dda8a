"""Dense ops on states so large that every workgroup of the matrix-core kernel
runs several blocks of columns (prefetch of the next block, both LDS buffers and
all three column slots in use), on both sides of each line of its launch rule for a
chip of 256 CUs, against the vector kernel on the device. A row is a sum of
2 * 2^k products on either side, each within 128 units in the last place in
the worst case and a few on average, as in the comparison with the FP64 applier."""
import numpy as np
import pytest

from qevedo.simulator import StateVector, library, lower_gates

pytestmark = pytest.mark.gpu


def unitary(seed, k):
    r = np.random.Generator(np.random.PCG64(seed))
    a = r.normal(size=(1 << k, 1 << k)) + 1j * r.normal(size=(1 << k, 1 << k))
    return np.linalg.qr(a)[0]


@pytest.mark.parametrize("precision,n,targets,controls", [
    ("double", 23, [0, 1, 2], []), ("double", 25, [2, 0, 22], [(1, True)]),  # 4 blocks a workgroup
    ("double", 24, [3, 1, 0, 2], []), ("double", 26, [1, 25, 0, 13], [(4, False), (9, True)]),
    ("double", 24, [4, 3, 2, 1, 0], []), ("double", 22, [0, 4, 8, 12, 16, 20], []),
    ("single", 24, [0, 1, 2, 3, 4], []), ("single", 27, [26, 0, 3, 9, 1], []),
    ("single", 22, [5, 4, 3, 2, 1, 0], []), ("single", 26, [0, 1, 2, 3, 4, 5], []),
    ("single", 27, [0, 4, 9, 14, 18, 23], [(1, True)]), ("single", 26, [25, 24, 23, 2, 1, 0], []),
    ("single", 8, [0, 1, 2, 3, 4], [(5, True)]), ("single", 6, [3, 5, 0, 4, 1, 2], []),  # fewer columns than a block
])
def test_against_the_vector_kernel(precision, n, targets, controls):
    state = lower_gates(library.random_circuit(n, 2, 5))
    op = [(targets, controls, unitary(n, len(targets)))]
    with StateVector(n, precision) as a, StateVector(n, precision) as b:
        for sv, vector in ((a, False), (b, True)):
            sv.apply_ops(state)
            sv.apply_ops(op, len(targets), None, dense_valu=vector)
        assert a.compare(b)["rel_l2"] < (3e-6 if precision == "single" else 3e-14)


@pytest.mark.parametrize("precision,n", [("single", 25), ("single", 26), ("single", 27), ("double", 25), ("double", 26)])
@pytest.mark.parametrize("targets,controls", [([1], [(0, True)]), ([24], []), ([0, 3], []), ([7, 2], [(24, False)]),
                                              ([1, 3, 5], []), ([23, 0, 12], [(1, True)]), ([9, 4, 7, 2], [])])
def test_vector_kernel_on_large_states(precision, n, targets, controls):
    """Sizes on both sides of the lines (512 MiB, 1 GiB) at which the vector
    kernel's launches change, against the stage kernel on the device."""
    state = lower_gates(library.random_circuit(n, 2, 5))
    u = unitary(n, len(targets))
    with StateVector(n, precision) as a, StateVector(n, precision) as b:
        a.apply_ops(state)
        a.apply(u, targets, controls)
        a.apply_ops([(targets, controls, u)], len(targets), None)
        b.apply_ops(state)
        b.apply_ops([(targets, controls, u)])
        b.apply_ops([(targets, controls, u)])
        assert a.compare(b)["rel_l2"] < (3e-6 if precision == "single" else 3e-14)

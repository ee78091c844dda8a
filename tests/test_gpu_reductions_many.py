"""Reductions beyond one page, one submission or one wave: Pauli strings by the
hundreds and thousands (X parts that straddle a submission), groups of every width
in one call, and <Z>, <ZZ> of states with more segments than a wave walks."""
import numpy as np
import pytest

from helpers import random_state, rng
from qevedo.simulator import Batch, StateVector, lower_gates

pytestmark = pytest.mark.gpu


def small_calls(sv, x, z):
    return np.concatenate([sv.expect_pauli(x[i:i + 9], z[i:i + 9]) for i in range(0, len(x), 9)])


@pytest.mark.parametrize("n,count", [(10, 512), (10, 513), (10, 5000), (13, 4100)])
@pytest.mark.parametrize("precision", ["single", "double"])
def test_many_strings(n, count, precision):
    """Sums of 2^n products of amplitudes, at most 1 in all: below 1e-12 apart in any order."""
    r = np.random.Generator(np.random.PCG64(count))
    xs = r.integers(0, 1 << n, count // 7)
    x = [int(v) for v in r.choice(xs, count)]
    z = [int(v) for v in r.integers(0, 1 << n, count)]
    with StateVector(n, precision) as sv:
        sv.set_amplitudes(random_state(rng(n), n))
        assert np.max(np.abs(sv.expect_pauli(x, z) - small_calls(sv, x, z))) < 1e-12


@pytest.mark.parametrize("n", [12, 17, 21])
@pytest.mark.parametrize("narrow", [0, 3, 40])
def test_groups_of_every_width(n, narrow):
    r = np.random.Generator(np.random.PCG64(n + narrow))
    x, z = [], []
    for part, width in [(0, 16), (0, 5), (3, 8), (1 << (n - 1), 3), (6, 2)] + [(8 + i, 1) for i in range(narrow)]:
        x += [part] * width
        z += [int(v) for v in r.integers(0, 1 << n, width)]
    order = r.permutation(len(x))
    x, z = [x[i] for i in order], [z[i] for i in order]
    with StateVector(n, "double") as sv:
        sv.set_amplitudes(random_state(rng(n), n))
        assert np.max(np.abs(sv.expect_pauli(x, z) - small_calls(sv, x, z))) < 1e-12


@pytest.mark.parametrize("n,precision,tol", [(24, "single", 1e-5), (25, "single", 1e-5), (26, "double", 1e-12)])
def test_z_of_many_segments(n, precision, tol):
    """A product of rx(t_q)|0>: <Z_q> = cos t_q. Two roundings of a factor per qubit."""
    t = 0.1 + 0.11 * np.arange(n)
    with StateVector(n, precision) as sv:
        sv.apply_ops(lower_gates([("rx", (q,), (float(t[q]),)) for q in range(n)]))
        z, zz = sv.expect_z()
    c = np.cos(t)
    assert np.max(np.abs(z - c)) < tol and np.max(np.abs(zz - c[:-1] * c[1:])) < tol


@pytest.mark.parametrize("n,precision,tol", [(5, "double", 1e-12), (14, "single", 1e-5), (17, "double", 1e-12)])
def test_batch_of_one_circuit(n, precision, tol):
    t = 0.1 + 0.11 * np.arange(n)
    batch = Batch([(n, lower_gates([("rx", (q,), (float(t[q]),)) for q in range(n)]))], precision)
    (z, zz), = batch.run()
    batch.close()
    c = np.cos(t)
    assert np.max(np.abs(z - c)) < tol and np.max(np.abs(zz - c[:-1] * c[1:])) < tol

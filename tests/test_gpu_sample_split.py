"""Sampling where its split changes: one lane per chunk (10 qubits; a state of
less than a batch), one batch per chunk (11), one chunk (15), 4 and 512 of them in
complex64, and the same in complex128 (chunks of 2^14), against the restated
two-pass sampler on the same amplitudes. Outcomes are whole numbers: equal."""
import numpy as np
import pytest

from helpers import random_state, rng
from oracle import oracle
from qevedo.simulator import StateVector

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,precision", [(10, "single"), (11, "single"), (15, "single"), (17, "single"), (24, "single"),
                                         (11, "double"), (14, "double"), (16, "double"), (23, "double")])
@pytest.mark.parametrize("kind", ["dense", "half"])
def test_outcomes(n, precision, kind):
    psi = random_state(rng(n), n)
    if kind == "half":  # chunks and blocks without probability, the last one among them
        psi[len(psi) // 2:] = 0
        psi[: len(psi) // 8] = 0
        psi /= np.linalg.norm(psi)
    with StateVector(n, precision) as sv, oracle.OracleState(n, precision) as o:
        sv.set_amplitudes(psi)
        o.set_amplitudes(sv.amplitudes())
        for u in (np.array([0.0]), np.array([1 - 2.0 ** -53]), rng(1).random(1),
                  np.concatenate([[0.0, 1 - 2.0 ** -53, 0.5, 5e-324], rng(2).random(5000)])):
            assert np.array_equal(sv.sample(u), o.sample(u))

"""Sampling at every number of chunks per workgroup of the chain kernel (4, 8 and 16:
25 and 26 qubits in complex64, 24 to 26 in complex128; the smaller and larger numbers
run on smaller and larger states), against the restated two-pass sampler on the
same amplitudes. Outcomes are whole numbers: equal."""
import numpy as np
import pytest

from helpers import random_state, rng
from oracle import oracle
from qevedo.simulator import StateVector

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,precision", [(25, "single"), (26, "single"), (24, "double"), (25, "double"), (26, "double")])
@pytest.mark.parametrize("kind", ["dense", "half"])
def test_outcomes(n, precision, kind):
    print(f"chunks per workgroup: {n} qubits {precision} {kind}", flush=True)
    part = random_state(rng(n), 18) * 2.0 ** (-(n - 18) / 2)
    psi = np.tile(part, 1 << (n - 18))
    psi[::1 << 18] *= 1 + 0.25 * np.arange(1 << (n - 18)) / (1 << (n - 18))  # chunks differ
    if kind == "half":  # chunks, and whole workgroups of them, without probability
        psi[len(psi) // 2:] = 0
        psi[len(psi) // 16: len(psi) // 16 + (3 << 15)] = 0
    psi /= np.linalg.norm(psi)
    with StateVector(n, precision) as sv, oracle.OracleState(n, precision) as o:
        sv.set_amplitudes(psi)
        o.set_amplitudes(sv.amplitudes())
        for u in (np.array([0.0, 1 - 2.0 ** -53]), np.concatenate([[0.0, 0.5, 5e-324], rng(2).random(3000)])):
            assert np.array_equal(sv.sample(u), o.sample(u))

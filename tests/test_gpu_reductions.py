"""The FP64 reductions at the sizes where their split changes, against NumPy in
64 bits on the amplitudes the device holds. Each value is a sum of terms whose
magnitudes add up to at most 1, so any order of a tree or of runs of at most
2^10 terms is within 2^11 roundings of 2^-53: 1e-12 is a bound for all."""
import numpy as np
import pytest

from helpers import random_state, rng
from qevedo.simulator import Batch, StateVector, library, lower_gates

pytestmark = pytest.mark.gpu
TOL = 1e-12


def loaded(n, precision):
    sv = StateVector(n, precision)
    sv.set_amplitudes(random_state(rng(400 + n), n))
    return sv, sv.amplitudes()


@pytest.mark.parametrize("precision", ["single", "double"])
@pytest.mark.parametrize("n", [1, 2, 5, 6, 7, 9, 10, 11, 16, 17, 18, 19, 22])
def test_z_norm_and_probabilities(n, precision):
    sv, a = loaded(n, precision)
    with sv:
        p = np.abs(a) ** 2
        z, zz = sv.expect_z()
        for q in range(n):
            t = p.reshape(-1, 2, 1 << q).sum(axis=(0, 2))
            assert abs(z[q] - (t[0] - t[1])) < TOL, q
            assert abs(sv.probability_one(q) - t[1]) < TOL, q
        for q in range(n - 1):
            t = p.reshape(-1, 2, 2, 1 << q).sum(axis=(0, 3))
            assert abs(zz[q] - (t[0, 0] + t[1, 1] - t[0, 1] - t[1, 0])) < TOL, q
        assert abs(sv.norm_sqr() - p.sum()) < TOL


@pytest.mark.parametrize("precision", ["single", "double"])
@pytest.mark.parametrize("n", [1, 4, 11, 12, 17, 21])
def test_pauli_groups(n, precision):
    """X parts with their highest bit low, in the middle and at the top, groups
    of 1 to 33 strings per X part (more than one pass takes), all at once."""
    r = rng(500 + n)
    sv, a = loaded(n, precision)
    xs, zs = [], []
    for x in {0, 1, (1 << n) - 1, 1 << (n - 1), (1 << (n // 2 + 1)) - 1}:
        if x < 1 << n:
            count = int(r.integers(1, 34))
            xs += [x] * count
            zs += [int(v) for v in r.integers(0, 1 << n, count)]
    order = r.permutation(len(xs))
    xs, zs = [xs[i] for i in order], [zs[i] for i in order]
    i = np.arange(1 << n, dtype=np.uint64)
    with sv:
        got = sv.expect_pauli(xs, zs)
    for t, (x, z) in enumerate(zip(xs, zs)):
        sign = np.zeros(1 << n, dtype=np.int64)
        for q in range(n):
            if z >> q & 1:
                sign ^= ((i >> np.uint64(q)) & np.uint64(1)).astype(np.int64)
        # P|j> = i^popcount(x & z) (-1)^popcount(j & z) |j ^ x>
        value = (1j) ** bin(x & z).count("1") * np.sum(np.conj(a[i ^ np.uint64(x)]) * a * (1 - 2 * sign))
        assert abs(got[t] - value.real) < TOL, (x, z)


@pytest.mark.parametrize("precision", ["single", "double"])
@pytest.mark.parametrize("n,qubit", [(1, 0), (5, 4), (13, 0), (14, 3), (15, 14), (18, 9)])
def test_measure_and_reset(n, qubit, precision):
    real = np.float32 if precision == "single" else np.float64
    for outcome in (0, 1):
        for reset in (False, True):
            sv, a = loaded(n, precision)
            with sv:
                p1 = sv.probability_one(qubit)
                u = p1 * 0.5 if outcome else p1 + (1 - p1) * 0.5
                if reset:
                    sv.reset(qubit, u)
                else:
                    assert sv.measure(qubit, u) == outcome
                keep = real(1.0 / np.sqrt(p1 if outcome else 1 - p1))
                v = a.reshape(-1, 2, 1 << qubit)
                want = np.zeros_like(v)
                to = 0 if reset else outcome
                want[:, to].real = (v[:, outcome].real.astype(real) * keep)
                want[:, to].imag = (v[:, outcome].imag.astype(real) * keep)
                assert np.array_equal(sv.amplitudes(), want.reshape(-1))


@pytest.mark.parametrize("sizes", [[15], [3, 17, 14, 21]])
def test_batch_values(sizes):
    gates = [library.hardware_efficient_ansatz(n, 2, 7 + n) for n in sizes]
    with Batch([(n, lower_gates(g)) for n, g in zip(sizes, gates)], "double") as b:
        for (z, zz), n, g in zip(b.run(), sizes, gates):
            with StateVector(n, "double") as sv:
                sv.apply_ops(lower_gates(g))
                wz, wzz = sv.expect_z()
            assert np.max(np.abs(z - wz)) < TOL
            assert zz.size == n - 1 and (n == 1 or np.max(np.abs(zz - wzz)) < TOL)


def test_lanes_of_destroyed_handles():
    """More handles at once than are kept for reuse, from several threads, each
    measuring its own state: no result reaches another handle's caller."""
    import threading

    wrong = []

    def work(seed):
        for i in range(6):
            svs = [StateVector(4 + (seed + k) % 5, "double") for k in range(3)]
            for k, sv in enumerate(svs):
                a = random_state(rng(100 * seed + 10 * i + k), sv.num_qubits)
                sv.set_amplitudes(a)
                p = np.abs(a.reshape(-1, 2, 2)[:, 1]) ** 2
                if abs(sv.probability_one(1) - p.sum()) > TOL or abs(sv.norm_sqr() - 1) > TOL:
                    wrong.append((seed, i, k))
            for sv in svs:
                sv.close()

    threads = [threading.Thread(target=work, args=(s,)) for s in range(5)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not wrong


@pytest.mark.parametrize("precision,tol", [("single", 1e-6), ("double", 1e-14)])
@pytest.mark.parametrize("k,controls", [(1, 0), (1, 2), (2, 0), (2, 1), (3, 0), (3, 1)])
def test_single_gates_by_argument(k, controls, precision, tol):
    """A gate by itself on high, low and controlled qubits against the dense
    product: 2^k complex products and sums of numbers below 1, 34 roundings."""
    from helpers import full_operator, random_unitary

    n = 7
    r = rng(60 + k)
    for qubits in (list(range(k + controls)), list(range(n - k - controls, n))[::-1], [3, 0, 6, 2, 5][: k + controls]):
        m = random_unitary(r, k)
        a = random_state(r, n)
        t, c = qubits[:k], qubits[k:]
        with StateVector(n, precision) as sv:
            sv.set_amplitudes(a)
            start = sv.amplitudes()
            sv.apply(m, t, [(q, j % 2 == 0) for j, q in enumerate(c)])
            got = sv.amplitudes()
        want = full_operator(n, m, t) @ start
        i = np.arange(1 << n)
        on = np.ones(1 << n, dtype=bool)
        for j, q in enumerate(c):
            on &= ((i >> q) & 1) == (1 if j % 2 == 0 else 0)
        assert np.max(np.abs(got - np.where(on, want, start))) < tol

"""Observables of one to hundreds of Pauli words on circuits of at most 12
qubits, on both sides of the line between the whole-circuit launch (one to 16
amplitudes a thread) and the general path, whose kernels the profile names;
against the oracle at the tolerances of the other adjoint tests, and batched
circuits likewise."""
import numpy as np
import pytest

import oracle as O
from helpers import random_hamiltonian, random_ops, random_state, to_capi, to_oracle

pytestmark = pytest.mark.gpu
NAMES = ["RX", "RY", "RZ", "CNOT", "CRX"]
TOL = [(np.complex128, 1e-10, 1e-12), (np.complex64, 0.0, 1e-5)]


def circuit(n, rng):
    names = NAMES if n > 1 else NAMES[:3]
    ops = random_ops(n, 25, rng, names=names)
    return ops, list(range(sum(1 for p in ops[1] if p)))


def scaled_hamiltonian(n, words, rng):
    """Coefficients that keep the energy of order one."""
    kind, coeffs, terms = random_hamiltonian(n, words, rng)
    return kind, [c / np.sqrt(words) for c in coeffs], terms


@pytest.mark.parametrize("dtype,rtol,atol", TOL)
@pytest.mark.parametrize("n", [1, 2, 5, 7, 8, 9, 10, 11, 12])
@pytest.mark.parametrize("words", [1, 2, 3, 33])
def test_few_words(capi, n, words, dtype, rtol, atol):
    rng = np.random.default_rng(100 * n + words)
    ops, tp = circuit(n, rng)
    obs = [scaled_hamiltonian(n, words, rng), ("named", "PauliZ", [0])]
    psi = random_state(n, rng).astype(dtype)
    s = capi.State(n, dtype)
    s.upload(psi)
    capi.profiling_enable(True)
    try:
        got = capi.adjoint_jacobian(s, [to_capi(capi, o) for o in obs], capi.Ops(*ops), tp, True)
        assert "circuit_sweep" in capi.profiling_names()
    finally:
        capi.profiling_enable(False)
    ref = O.adjoint_jacobian(psi.astype(np.complex128), [to_oracle(o) for o in obs], O.Ops(*ops), tp, True)
    np.testing.assert_allclose(got, ref, rtol=rtol, atol=atol)


@pytest.mark.parametrize("dtype,rtol,atol", TOL)
@pytest.mark.parametrize("n,words,n_obs,whole", [(8, 300, 1, True), (8, 1200, 1, False), (10, 600, 1, False),
                                                 (10, 300, 3, False), (12, 600, 1, False), (12, 600, 2, False),
                                                 (12, 90, 3, True)])
def test_many_words(capi, n, words, n_obs, whole, dtype, rtol, atol):
    rng = np.random.default_rng(100 * n + words)
    ops, tp = circuit(n, rng)
    obs = [scaled_hamiltonian(n, words, rng) for _ in range(n_obs)]
    s = capi.State(n, dtype)
    capi.profiling_enable(True)
    try:
        got = capi.adjoint_jacobian(s, [to_capi(capi, o) for o in obs], capi.Ops(*ops), tp, True)
        # Three observables of 300 words: on either side by the precision (8 or 16 amplitudes a thread).
        assert ("circuit_sweep" in capi.profiling_names()) == (whole or (dtype == np.complex128 and n_obs == 3))
    finally:
        capi.profiling_enable(False)
    ref = O.adjoint_jacobian(O.zero_state(n), [to_oracle(o) for o in obs], O.Ops(*ops), tp, True)
    np.testing.assert_allclose(got, ref, rtol=rtol, atol=atol)


@pytest.mark.parametrize("dtype,rtol,atol", TOL)
def test_batched_words(capi, monkeypatch, dtype, rtol, atol):
    rng = np.random.default_rng(17)
    sizes = [1, 4, 8, 9, 10, 11, 12, 13, 14]
    circuits = [circuit(n, rng) for n in sizes]
    obs = [scaled_hamiltonian(n, 40, rng) for n in sizes]
    for whole in ("10", ""):
        monkeypatch.setenv("PLK_BATCH_WHOLE_QUBITS", whole)
        values, rows = capi.adjoint_batched(sizes, [capi.Ops(*o) for o, _ in circuits],
                                            [to_capi(capi, o) for o in obs], [tp for _, tp in circuits], dtype=dtype)
        for n, (ops, tp), ob, v, row in zip(sizes, circuits, obs, values, rows):
            o = O.Ops(*ops)
            np.testing.assert_allclose(v, O.expval(O.apply_ops(O.zero_state(n), o), to_oracle(ob)), rtol=rtol, atol=atol)
            np.testing.assert_allclose(row, O.adjoint_jacobian(O.zero_state(n), [to_oracle(ob)], o, tp, True)[0],
                                       rtol=rtol, atol=atol)

"""Batched calls that differ in one matrix, of an op or of an observable's
wires, coefficients or order, plan anew: values against the oracle, each
set of handles called twice."""
import numpy as np
import pytest

import oracle as O
from helpers import random_unitary, to_capi, to_oracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype,rtol,atol", [(np.complex128, 1e-10, 1e-12), (np.complex64, 0.0, 1e-5)])
def test_matrices_and_observables_are_part_of_the_plan(capi, dtype, rtol, atol):
    rng = np.random.default_rng(8)
    n = 3
    one, two = random_unitary(2, rng), random_unitary(4, rng)
    z, x = ("named", "PauliZ", [0]), ("named", "PauliX", [1])
    variants = [(a, b, o) for a, b in ((one, two), (one.conj(), two), (one, two.T), (two[:2, :2], two))
                for o in (("ham", [1.0, 0.5], [z, x]), ("ham", [0.5, 1.0], [z, x]), ("ham", [1.0, 0.5], [x, z]))]
    variants += variants[:2]
    for a, b, ob in variants:
        if not np.allclose(a.conj().T @ a, np.eye(2)):
            a, _ = np.linalg.qr(a)
        ops = (["RX", "U1", "RY", "U2", "RZ"], [[0.3], [], [0.4], [], [0.5]], [[0], [0], [1], [0, 1], [1]], [False] * 5,
               [[], a.reshape(-1), [], b.reshape(-1), []])
        handle, obs = capi.Ops(*ops), to_capi(capi, ob)
        o = O.Ops(*ops)
        for _ in range(2):
            values, rows = capi.adjoint_batched([n], [handle], [obs], [[0, 1, 2]], dtype=dtype)
            np.testing.assert_allclose(values[0], O.expval(O.apply_ops(O.zero_state(n), o), to_oracle(ob)), rtol=rtol,
                                       atol=atol)
            np.testing.assert_allclose(rows[0], O.adjoint_jacobian(O.zero_state(n), [to_oracle(ob)], o, [0, 1, 2], True)[0],
                                       rtol=rtol, atol=atol)

"""Jacobians of op lists in which a matrix on three to five wires that is not
unitary stands between trainable gates of other wires: the derivatives before and
after it differ, so no run of gates reaches over it. Against the oracle
(AdjointDiffKokkos.hpp:432-470 gate by gate) at the tolerances of the other
adjoint tests; the same with a unitary one, over which runs may reach."""
import numpy as np
import pytest

import oracle as O
from helpers import random_state, random_unitary, to_capi, to_oracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype,rtol,atol", [(np.complex128, 1e-10, 1e-12), (np.complex64, 0.0, 1e-5)])
@pytest.mark.parametrize("n", [6, 9, 13])
@pytest.mark.parametrize("m", [3, 4, 5])
@pytest.mark.parametrize("unitary", [False, True])
def test_jacobian(capi, unitary, m, n, dtype, rtol, atol):
    rng = np.random.default_rng(100 * m + n)
    names, params, wires, mats = [], [], [], []

    def add(name, w, angle=None, matrix=()):
        names.append(name)
        params.append([] if angle is None else [angle])
        wires.append([int(x) for x in w])
        mats.append(list(matrix))

    for layer in range(3):
        for w in range(n):
            add(["RX", "RY", "RZ"][(w + layer) % 3], [w], rng.uniform(0, 2 * np.pi))
        M = random_unitary(2**m, rng)
        if not unitary:
            M = M * rng.uniform(0.6, 1.0, size=(2**m, 1))
        add("QubitUnitary", rng.choice(n, size=m, replace=False), None, M.reshape(-1))
        for w in range(n):
            add(["RY", "RZ", "RX"][(w + layer) % 3], [w], rng.uniform(0, 2 * np.pi))
        for w in range(0, n - 1, 2):
            add("CNOT", [w, w + 1])
    ops = (names, params, wires, [bool(rng.integers(2)) for _ in names], mats)
    obs = [("named", "PauliZ", [0]), ("ham", [0.3, 0.8], [("named", "PauliX", [n - 1]), ("named", "PauliY", [n // 2])])]
    tp = list(range(sum(1 for p in params if p)))
    psi = random_state(n, rng).astype(dtype)
    s = capi.State(n, dtype)
    s.upload(psi)
    got = capi.adjoint_jacobian(s, [to_capi(capi, o) for o in obs], capi.Ops(*ops), tp, True)
    ref = O.adjoint_jacobian(psi.astype(np.complex128), [to_oracle(o) for o in obs], O.Ops(*ops), tp, True)
    np.testing.assert_allclose(got, ref, rtol=rtol, atol=atol)

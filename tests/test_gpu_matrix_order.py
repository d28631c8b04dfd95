"""Jacobians of op lists with matrices that are not unitary among trainable
gates. The reverse sweep applies their conjugate transposes to the state and to
every H lambda, so an entry depends on which of them have been applied before
it, on any wire: fused runs and passes keep that order. At sizes of every
reverse path, against the oracle (AdjointDiffKokkos.hpp:432-470 gate by gate) at
the tolerances of the other adjoint tests."""
import numpy as np
import pytest

import oracle as O
from helpers import random_state, to_capi, to_oracle
from test_gpu_matrix_scale import scaled_circuit

pytestmark = pytest.mark.gpu

# Norms of at most one, so that entries stay of order one.
CONTRACTIONS = {
    "scaled": [0.75, 0, 0, 0.75],
    "projector": [1, 0, 0, 0],
    "plus projector": [0.5, 0.5, 0.5, 0.5],
    "lopsided": [0.4, 0.2j, -0.3, 0.8],
    "zero": [0, 0, 0, 0],
}


@pytest.mark.parametrize("dtype,rtol,atol", [(np.complex128, 1e-10, 1e-12), (np.complex64, 0.0, 1e-5)])
@pytest.mark.parametrize("n", [5, 8, 9, 12, 13, 17])
@pytest.mark.parametrize("kind", sorted(CONTRACTIONS))
def test_jacobian(capi, kind, n, dtype, rtol, atol):
    rng = np.random.default_rng(37 * n + len(kind))
    ops = scaled_circuit(n, CONTRACTIONS[kind], rng)
    obs = [("named", "PauliZ", [0]), ("ham", [0.3, 0.8], [("named", "PauliX", [n - 1]), ("named", "PauliY", [n // 2])])]
    tp = list(range(sum(1 for p in ops[1] if p)))
    psi = random_state(n, rng).astype(dtype)
    for apply in (True, False):
        s = capi.State(n, dtype)
        s.upload(psi)
        got = capi.adjoint_jacobian(s, [to_capi(capi, o) for o in obs], capi.Ops(*ops), tp, apply)
        ref = O.adjoint_jacobian(psi.astype(np.complex128), [to_oracle(o) for o in obs], O.Ops(*ops), tp, apply)
        np.testing.assert_allclose(got, ref, rtol=rtol, atol=atol)

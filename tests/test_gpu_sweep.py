"""Whole circuits in one launch (states of at most 12 qubits): states smaller
than a tile, of exactly one tile and of several, both precisions, with more
sums than one pass holds, against the oracle and against the pass-by-pass path
(PLK_SWEEP=0). Tolerances as in the other adjoint tests."""
import numpy as np
import pytest

import oracle as O
from helpers import GATES, random_hamiltonian, random_ops, random_state, to_capi, to_oracle

pytestmark = pytest.mark.gpu

ONE_TWO_WIRE = [g for g in GATES if g != "Identity" and GATES[g][0] in (1, 2) and GATES[g][1] <= 1]


@pytest.mark.parametrize("dtype,rtol,atol", [(np.complex128, 1e-10, 1e-12), (np.complex64, 0.0, 1e-5)])
@pytest.mark.parametrize("n", [1, 2, 3, 6, 8, 9, 10, 11, 12])
@pytest.mark.parametrize("apply", [True, False])
def test_small_circuits(monkeypatch, n, dtype, rtol, atol, apply):
    from pennylane_lightning_kokkos_amd import _capi

    rng = np.random.default_rng(40 * n + apply)
    names = [g for g in ONE_TWO_WIRE if GATES[g][0] <= n]
    ops = random_ops(n, 150, rng, names=names, with_matrix=n > 2)
    if any(len(w) > 2 for w in ops[2]):  # the matrix op stays on two wires
        k = [len(w) > 2 for w in ops[2]].index(True)
        ops = tuple(x[:k] + x[k + 1:] for x in ops)
    npar = sum(1 for p in ops[1] if p)
    tp = sorted(int(t) for t in rng.choice(npar, max(1, npar - 3), replace=False))
    obs = [random_hamiltonian(n, 6, rng), ("named", "PauliY", [n - 1]), ("named", "Hadamard", [0])]
    psi = random_state(n, rng).astype(dtype)
    cops, cobs = _capi.Ops(*ops), [to_capi(_capi, o) for o in obs]

    def jacobian():
        s = _capi.State(n, dtype)
        s.upload(psi)
        out = _capi.adjoint_jacobian(s, cobs, cops, tp, apply)
        assert np.array_equal(s.download(), psi)  # the input state is left as it was
        return out

    got = jacobian()
    ref = O.adjoint_jacobian(psi.astype(np.complex128), [to_oracle(o) for o in obs], O.Ops(*ops), tp, apply)
    np.testing.assert_allclose(got, ref, rtol=rtol, atol=atol)
    assert np.array_equal(got, jacobian())
    monkeypatch.setenv("PLK_SWEEP", "0")
    np.testing.assert_allclose(jacobian(), got, rtol=rtol, atol=atol)
    monkeypatch.delenv("PLK_SWEEP")
    s = _capi.State(n, dtype)
    s.upload(psi)
    s.apply_ops(cops)
    np.testing.assert_allclose(s.download(), O.apply_ops(psi.astype(np.complex128), O.Ops(*ops)), rtol=0,
                               atol=1e-12 if dtype == np.complex128 else 2e-5)

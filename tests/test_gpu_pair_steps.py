"""Single-op steps on two-state subspaces (SingleExcitation, DoubleExcitation,
CNOT, CRX and phases between them) with 1 to 9 observables, alternating with
register-tile passes, at sizes below and above the graph limit's old and new
places, replayed and eager, against the oracle (tolerances as elsewhere)."""
import numpy as np
import pytest

import oracle as O
from helpers import random_hamiltonian, random_state, to_capi, to_oracle

pytestmark = pytest.mark.gpu


def ansatz(n, rng, rounds):
    names, params, wires = [], [], []
    for _ in range(rounds):
        for name, m in (("DoubleExcitation", 4), ("SingleExcitation", 2), ("DoubleExcitation", 4), ("CNOT", 2),
                        ("Toffoli", 3), ("CRX", 2), ("CZ", 2), ("DoubleExcitation", 4), ("RX", 1), ("CNOT", 2)):
            names.append(name)
            params.append([] if name in ("CNOT", "CZ", "Toffoli") else [float(rng.uniform(0, 2 * np.pi))])
            wires.append([int(w) for w in rng.choice(n, m, replace=False)])
    return names, params, wires, [bool(rng.integers(2)) for _ in names], [[] for _ in names]


@pytest.mark.parametrize("dtype,rtol,atol", [(np.complex128, 1e-10, 1e-12), (np.complex64, 0.0, 1e-5)])
@pytest.mark.parametrize("n,n_obs,rounds", [(9, 1, 3), (11, 9, 2), (13, 2, 3), (14, 8, 2), (19, 3, 1)])
def test_pair_steps(n, n_obs, rounds, dtype, rtol, atol):
    from pennylane_lightning_kokkos_amd import _capi

    rng = np.random.default_rng(100 * n + n_obs)
    ops = ansatz(n, rng, rounds)
    npar = sum(1 for p in ops[1] if p)
    obs = [random_hamiltonian(n, 3, rng)] + [("named", "PauliZ", [w]) for w in range(n_obs - 1)]
    psi = random_state(n, rng).astype(dtype)
    s = _capi.State(n, dtype)
    s.upload(psi)
    cobs, cops = [to_capi(_capi, o) for o in obs], _capi.Ops(*ops)
    ref = O.adjoint_jacobian(psi.astype(np.complex128), [to_oracle(o) for o in obs], O.Ops(*ops), list(range(npar)),
                             True)
    calls = [_capi.adjoint_jacobian(s, cobs, cops, list(range(npar)), True) for _ in range(3)]
    for got in calls:  # eager, captured, replayed
        np.testing.assert_allclose(got, ref, rtol=rtol, atol=atol)
    assert np.array_equal(calls[1], calls[2])
    s.apply_ops(cops)
    np.testing.assert_allclose(s.download(), O.apply_ops(psi.astype(np.complex128), O.Ops(*ops)), rtol=0,
                               atol=1e-12 if dtype == np.complex128 else 2e-5)

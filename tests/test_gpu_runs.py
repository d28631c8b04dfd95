"""Fused one-wire runs in register-tile passes: chains of trainable and fixed
one-wire gates between two-wire gates, on every wire, so that a pass mixes all
of its tile bits (each register and lane position is exchanged), with the
Jacobian of every gate of a run formed from the run's Pauli sums. Against the
oracle at 1e-10 relative (complex128) and 1e-5 absolute (complex64), the
tolerances of the other adjoint tests."""
import numpy as np
import pytest

import oracle as O
from helpers import random_hamiltonian, random_state, to_capi, to_oracle

pytestmark = pytest.mark.gpu

CHAIN = ["RX", "RY", "RZ", "PhaseShift", "Hadamard", "S", "T", "PauliX", "PauliY", "PauliZ"]
PAIRS = ["CNOT", "CZ", "CRX", "IsingZZ", "SWAP", "ControlledPhaseShift", "SingleExcitation"]
PARAMETRIC = {"RX", "RY", "RZ", "PhaseShift", "CRX", "IsingZZ", "ControlledPhaseShift", "SingleExcitation"}


def chain_circuit(n, rng, layers=2):
    names, params, wires, inverses = [], [], [], []

    def add(name, w):
        names.append(name)
        params.append([float(rng.uniform(0, 2 * np.pi))] if name in PARAMETRIC else [])
        wires.append(w)
        inverses.append(bool(rng.integers(2)))

    for _ in range(layers):
        for w in rng.permutation(n):
            for _ in range(int(rng.integers(1, 5))):
                add(CHAIN[rng.integers(len(CHAIN))], [int(w)])
        for _ in range(n // 2):
            add(PAIRS[rng.integers(len(PAIRS))], [int(x) for x in rng.choice(n, 2, replace=False)])
    return names, params, wires, inverses, [[] for _ in names]


@pytest.mark.parametrize("dtype,rtol,atol", [(np.complex128, 1e-10, 1e-12), (np.complex64, 0.0, 1e-5)])
@pytest.mark.parametrize("n,n_obs", [(9, 3), (10, 1), (10, 4), (11, 1), (11, 2), (13, 5), (17, 3)])
def test_fused_runs_match_oracle(n, n_obs, dtype, rtol, atol):
    from pennylane_lightning_kokkos_amd import _capi

    rng = np.random.default_rng(1000 * n + n_obs)
    ops = chain_circuit(n, rng)
    npar = sum(1 for p in ops[1] if p)
    tp = sorted(int(t) for t in rng.choice(npar, max(1, 3 * npar // 4), replace=False))
    obs = [random_hamiltonian(n, 3, rng)] + [("named", "PauliZ", [w]) for w in range(n_obs - 1)]
    psi = random_state(n, rng).astype(dtype)
    s = _capi.State(n, dtype)
    s.upload(psi)
    got = _capi.adjoint_jacobian(s, [to_capi(_capi, o) for o in obs], _capi.Ops(*ops), tp, True)
    ref = O.adjoint_jacobian(psi.astype(np.complex128), [to_oracle(o) for o in obs], O.Ops(*ops), tp, True)
    np.testing.assert_allclose(got, ref, rtol=rtol, atol=atol)
    s.apply_ops(_capi.Ops(*ops))
    amps = O.apply_ops(psi.astype(np.complex128), O.Ops(*ops))
    np.testing.assert_allclose(s.download(), amps, rtol=0, atol=1e-12 if dtype == np.complex128 else 2e-5)

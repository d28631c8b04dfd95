"""Batched circuits with runs of one-wire gates whose matrices and Jacobian
coefficients are formed on the device from each call's angles: whole and
staged circuits (PLK_BATCH_WHOLE_QUBITS moves the line), new angles on a
resident plan including special ones (0, pi), against the oracle at the
tolerances of the other batched tests."""
import numpy as np
import pytest

import oracle as O
from helpers import random_hamiltonian, to_capi, to_oracle
from test_gpu_runs import PARAMETRIC, chain_circuit

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype,rtol,atol", [(np.complex128, 1e-10, 1e-12), (np.complex64, 0.0, 1e-5)])
@pytest.mark.parametrize("whole", ["", "10", "20"])
def test_batched_runs(monkeypatch, dtype, rtol, atol, whole):
    from pennylane_lightning_kokkos_amd import _capi

    if whole:
        monkeypatch.setenv("PLK_BATCH_WHOLE_QUBITS", whole)
    rng = np.random.default_rng(77)
    sizes = [2, 3, 9, 10, 11, 12, 13, 14, 15]
    circuits = [chain_circuit(n, rng) for n in sizes]
    for names, params, wires, _, mats in circuits:  # gates outside the patch: fixed by the plan
        names.append("MultiRZ")
        params.append([0.3])
        wires.append([0])
        mats.append([])
    circuits = [(a, b, c, d + [False], e) for a, b, c, d, e in circuits]
    obs = [random_hamiltonian(n, 4, rng) for n in sizes]
    trainable = []
    for ops in circuits:
        npar = sum(1 for p in ops[1] if p)
        trainable.append(sorted(int(t) for t in rng.choice(npar, max(1, npar - 2), replace=False)))
    for call in range(3):
        for ops in circuits:
            for k, name in enumerate(ops[0]):
                if name in PARAMETRIC and name in ("RX", "RY", "RZ", "PhaseShift"):
                    ops[1][k] = [float(rng.uniform(0, 2 * np.pi)) if call < 2 else float(rng.choice([0.0, np.pi]))]
        values, rows = _capi.adjoint_batched(sizes, [_capi.Ops(*ops) for ops in circuits],
                                             [to_capi(_capi, o) for o in obs], trainable, dtype=dtype)
        for n, ops, ob, tp, v, row in zip(sizes, circuits, obs, trainable, values, rows):
            ref = O.adjoint_jacobian(O.zero_state(n), [to_oracle(ob)], O.Ops(*ops), tp, True)[0]
            np.testing.assert_allclose(row, ref, rtol=rtol, atol=atol)
            psi = O.apply_ops(O.zero_state(n), O.Ops(*ops))
            s = _capi.State(n)
            s.upload(psi)
            assert abs(v - s.expval(to_capi(_capi, ob))) < (1e-11 if dtype == np.complex128 else 1e-5)

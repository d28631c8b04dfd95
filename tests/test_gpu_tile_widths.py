"""Register tiles of every width a plan chooses by the size of the state: on
both sides of each change, against the same circuit on the oracle (small states)
or against its smaller factor (large ones)."""
import numpy as np
import pytest

import oracle as O
from helpers import random_ops, random_state, to_capi, to_oracle

pytestmark = pytest.mark.gpu

GATES = ["RX", "RY", "RZ", "Hadamard", "PhaseShift", "S", "PauliY", "CNOT", "CZ", "CRX", "CRZ", "IsingXX", "IsingZZ",
         "SWAP", "SingleExcitation"]


# 1e-10 / 1e-5 for derivatives, 1e-12 / 2e-5 for amplitudes: the tolerances of
# the other tests of these kernels.
@pytest.mark.parametrize("dtype,jtol,atol", [(np.complex128, 1e-10, 1e-12), (np.complex64, 1e-5, 2e-5)])
@pytest.mark.parametrize("n,n_obs", [(9, 1), (13, 1), (13, 2), (16, 9), (18, 1), (19, 1)])
def test_small_states(capi, monkeypatch, n, n_obs, dtype, jtol, atol):
    monkeypatch.setenv("PLK_SWEEP", "0")
    rng = np.random.default_rng(10 * n + n_obs)
    ops = random_ops(n, 50 if n < 16 else 25, rng, names=GATES)
    psi = random_state(n, rng).astype(dtype)
    obs = [("named", "PauliZ", [j % n]) for j in range(n_obs)]
    tp = list(range(sum(1 for p in ops[1] if p)))
    s = capi.State(n, dtype)
    s.upload(psi)
    got = capi.adjoint_jacobian(s, [to_capi(capi, o) for o in obs], capi.Ops(*ops), tp, True)
    ref = O.adjoint_jacobian(psi.astype(np.complex128), [to_oracle(o) for o in obs], O.Ops(*ops), tp, True)
    np.testing.assert_allclose(got, ref, rtol=0, atol=jtol)
    s.apply_ops(capi.Ops(*ops))
    np.testing.assert_allclose(s.download(), O.apply_ops(psi.astype(np.complex128), O.Ops(*ops)), rtol=0, atol=atol)


@pytest.mark.parametrize("dtype,jtol,atol", [(np.complex128, 1e-10, 1e-12), (np.complex64, 1e-5, 2e-5)])
@pytest.mark.parametrize("n", [20, 21, 22, 23, 24])
def test_large_states(capi, n, dtype, jtol, atol):
    m = 10  # the circuit's wires, spread over the register; the others stay 0
    rng = np.random.default_rng(n)
    ops = random_ops(m, 120, rng, names=GATES)
    wires = sorted(int(w) for w in rng.choice(n, m, replace=False))
    large = (ops[0], ops[1], [[wires[w] for w in ws] for ws in ops[2]], ops[3], ops[4])
    tp = list(range(sum(1 for p in ops[1] if p)))
    s = capi.State(n, dtype)
    got = capi.adjoint_jacobian(s, [to_capi(capi, ("named", "PauliZ", [wires[3]]))], capi.Ops(*large), tp, True)
    ref = O.adjoint_jacobian(O.zero_state(m), [to_oracle(("named", "PauliZ", [3]))], O.Ops(*ops), tp, True)
    np.testing.assert_allclose(np.ravel(got), np.ravel(ref), rtol=0, atol=jtol)
    s.apply_ops(capi.Ops(*large))
    psi = s.download()
    index = np.zeros(2 ** m, np.int64)
    for w in range(m):
        index |= ((np.arange(2 ** m) >> (m - 1 - w)) & 1) << (n - 1 - wires[w])
    np.testing.assert_allclose(psi[index], O.apply_ops(O.zero_state(m), O.Ops(*ops)), rtol=0, atol=atol)
    assert abs(np.linalg.norm(psi[index]) - np.linalg.norm(psi)) < 1e-6

"""Register-tile plans that exchange tile bits for outside ones (calls that move
1 GiB a pass or more), against the oracle.

Such states are beyond the oracle's reach, so the large circuit is a product:
one circuit on the even wires and another on the odd ones, interleaved, and an
idle wire. Its amplitudes are products of the small circuits' amplitudes and the
derivatives of an observable on one half are those of that half's circuit."""
import numpy as np
import pytest

import oracle as O
from helpers import random_ops, to_capi, to_oracle

pytestmark = pytest.mark.gpu

GATES = ["RX", "RY", "RZ", "Hadamard", "PhaseShift", "CNOT", "CZ", "CRX", "CRZ", "IsingXX", "IsingZZ", "SWAP",
         "ControlledPhaseShift"]


def product_circuit(m, count, seed):
    """Two circuits on m wires and their interleaved product: wire w of the
    first is wire 2 w, of the second 2 w + 1."""
    rng = np.random.default_rng(seed)
    halves = [random_ops(m, count, rng, names=GATES) for _ in range(2)]
    both = ([], [], [], [], [])
    for k in range(count):
        for shift, half in enumerate(halves):
            for column, values in zip(both, half):
                column.append(values[k])
            both[2][-1] = [2 * w + shift for w in half[2][k]]
    return halves, both


# 300 gates on amplitudes below 1: 1e-12 as for every FP64 state.
def test_forward_product(capi):
    m, n = 12, 25
    halves, both = product_circuit(m, 150, 1)
    a, b = (O.apply_ops(O.zero_state(m), O.Ops(*h)) for h in halves)
    s = capi.State(n, np.complex128)
    s.apply_ops(capi.Ops(*both))
    psi = s.download()
    ia, ib = np.random.default_rng(2).integers(0, 2 ** m, (2, 5000))
    index = np.zeros(5000, np.int64)
    for w in range(m):
        index |= ((ia >> (m - 1 - w)) & 1) << (n - 1 - 2 * w)
        index |= ((ib >> (m - 1 - w)) & 1) << (n - 2 - 2 * w)
    np.testing.assert_allclose(psi[index], a[ia] * b[ib], rtol=0, atol=1e-12)
    assert abs(np.linalg.norm(psi) - 1) < 1e-12


# Tolerances of the other adjoint tests.
@pytest.mark.parametrize("dtype,n_obs,tol", [(np.complex128, 4, 1e-10), (np.complex64, 8, 1e-5)])
def test_jacobian_product(capi, dtype, n_obs, tol):
    m, n = 11, 23
    halves, both = product_circuit(m, 100, 5)
    sites = [(j % 2, j % m) for j in range(n_obs)]
    got = capi.adjoint_jacobian(capi.State(n, dtype),
                                [to_capi(capi, ("named", "PauliZ", [2 * w + h])) for h, w in sites],
                                capi.Ops(*both), list(range(sum(1 for p in both[1] if p))), True)
    ref = np.zeros(got.shape)
    columns = [[], []]  # the product's parameters of each half, in order
    count = 0
    for k, p in enumerate(both[1]):
        if p:
            columns[k % 2].append(count)
            count += 1
    for h in range(2):
        rows = [j for j in range(n_obs) if sites[j][0] == h]
        jac = O.adjoint_jacobian(O.zero_state(m), [to_oracle(("named", "PauliZ", [sites[j][1]])) for j in rows],
                                 O.Ops(*halves[h]), list(range(len(columns[h]))), True)
        ref[np.ix_(rows, columns[h])] = np.asarray(jac).reshape(len(rows), -1)
    np.testing.assert_allclose(np.asarray(got).reshape(ref.shape), ref, rtol=0, atol=tol)

"""Accuracy of complex64 op lists on states of at most 12 qubits.

200 unitary operations round each amplitude at most four times each (two
products and their sums, per part), by at most 6e-8 of its size, in directions
that do not depend on one another: a norm of 6e-8 sqrt(800) = 1.7e-6 for a
unit state."""
import numpy as np
import pytest

import oracle as O
from helpers import random_ops, random_state

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [5, 9, 12])
def test_small_forward_accuracy(capi, n):
    rng = np.random.default_rng(640 + n)
    ops = random_ops(n, 200, rng, names=["RX", "RY", "RZ", "CNOT", "CRY", "IsingXX", "DoubleExcitation"])
    psi = random_state(n, rng).astype(np.complex64)
    psi64 = psi.astype(np.complex128)
    s = capi.State(n, np.complex64)
    s.upload(psi)
    s.apply_ops(capi.Ops(*ops))
    want = O.apply_ops(psi64, O.Ops(*ops))
    assert np.linalg.norm(s.download() - want) <= 1.7e-6 * np.linalg.norm(psi64)

"""Op lists of one to ten operations on states that lists of more run whole in
one launch: both sides of that line, which the profile names, against the oracle
at the tolerances of the other forward tests."""
import numpy as np
import pytest

import oracle as O
from helpers import random_ops, random_state

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype,atol", [(np.complex128, 1e-12), (np.complex64, 2e-5)])
@pytest.mark.parametrize("n", [1, 2, 3, 4, 8, 9, 10, 12])
def test_short_lists(capi, n, dtype, atol):
    rng = np.random.default_rng(600 + n)
    names = ["RX", "RY", "RZ", "Hadamard", "CNOT", "CRX", "IsingXX"] if n > 1 else ["RX", "RY", "RZ", "Hadamard"]
    line = 8 if n <= 3 else 6 if dtype == np.complex64 else 4
    for count in range(1, 11):
        ops = random_ops(n, count, rng, names=names)
        psi = random_state(n, rng).astype(dtype)
        s = capi.State(n, dtype)
        s.upload(psi)
        capi.profiling_enable(True)
        try:
            s.apply_ops(capi.Ops(*ops))
            assert ("circuit_sweep" in capi.profiling_names()) == (count > line)
        finally:
            capi.profiling_enable(False)
        np.testing.assert_allclose(s.download(), O.apply_ops(psi.astype(np.complex128), O.Ops(*ops)), rtol=0, atol=atol)

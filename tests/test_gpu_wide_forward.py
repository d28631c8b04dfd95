"""complex64 forward passes computed in FP64 and rounded when a pass stores its
tile: the state is closer to the FP64 one than a rounding at every operation
leaves it."""
import numpy as np
import pytest

import oracle as O
from helpers import random_ops

pytestmark = pytest.mark.gpu


# 200 gates in at most 40 passes, each rounding an amplitude to 6e-8 relative
# once: 6e-8 * sqrt(40) = 3.8e-7 of the state's norm at most.
@pytest.mark.parametrize("n", [13, 16, 19])
def test_rounding_once_a_pass(capi, n):
    ops = random_ops(n, 200, np.random.default_rng(n), names=["RX", "RY", "RZ", "Hadamard", "CNOT", "CRX", "IsingXX"])
    s = capi.State(n, np.complex64)
    s.apply_ops(capi.Ops(*ops))
    ref = O.apply_ops(O.zero_state(n), O.Ops(*ops))
    assert np.linalg.norm(s.download() - ref) < 3.8e-7

"""Marginals on both sides of the state size from which bins of low wires are
summed together (4 MiB), and of one or several ranges a bin, against the oracle
(MeasuresKokkos.hpp:389-569)."""
import numpy as np
import pytest

import oracle as O
from helpers import random_state

pytestmark = pytest.mark.gpu


# 1e-12: sums of at most 2^20 products of FP64 rounding 1e-16 each, of total 1.
@pytest.mark.parametrize("dtype", [np.complex128, np.complex64])
@pytest.mark.parametrize("n", [8, 13, 18, 19, 20])
def test_marginals(capi, n, dtype):
    s = capi.State(n, dtype)
    s.upload(random_state(n, np.random.default_rng(190 + n)).astype(dtype))
    psi = s.download().astype(np.complex128)
    low = [n - 1 - k for k in range(7)]
    for wires in (low[:1], low[:2], low[:3], low[:4], low[:5], low[:6], low[::-1], [0], [0, low[1]], [low[2], 1, low[0]],
                  list(range(n - 7)), list(range(n - 6)), list(range(3, n - 3))):
        np.testing.assert_allclose(s.probs(wires), O.probs(psi, wires), rtol=0, atol=1e-12, err_msg=f"{wires}")

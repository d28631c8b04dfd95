"""A captured Jacobian whose observable chunks change between calls
(PLK_RTILE_NJ is read on each call) is captured again: the partial sums of the
launches and the entries that add them up follow the same layout."""
import numpy as np
import pytest

from helpers import random_ops, to_capi

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [14, 20])
def test_chunks_change_between_calls(capi, monkeypatch, n):
    rng = np.random.default_rng(n)
    ops = random_ops(n, 40, rng, names=["RX", "RY", "RZ", "CNOT", "CRX"])
    obs = [to_capi(capi, ("named", "PauliZ", [j])) for j in range(5)]
    cops = capi.Ops(*ops)
    tp = list(range(sum(1 for p in ops[1] if p)))
    s = capi.State(n, np.complex128)
    ref = np.asarray(capi.adjoint_jacobian(s, obs, cops, tp, True))
    for _ in range(2):
        for nj in ("2", "3", "1", "4"):
            monkeypatch.setenv("PLK_RTILE_NJ", nj)
            for _ in range(3):
                got = np.asarray(capi.adjoint_jacobian(s, obs, cops, tp, True))
                np.testing.assert_allclose(got, ref, rtol=0, atol=1e-12)

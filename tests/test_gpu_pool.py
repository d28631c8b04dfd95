"""Temporary states are recycled, also after a program has released more
evaluated observables than the table pool holds: a repeated Jacobian then
allocates nothing on the device."""
import numpy as np
import pytest

from helpers import random_ops, to_capi

pytestmark = pytest.mark.gpu


def test_released_observables_leave_states_recycled(capi, monkeypatch):
    monkeypatch.setenv("PLK_GRAPH", "0")
    monkeypatch.setenv("PLK_SWEEP", "0")
    n = 10
    ops = random_ops(n, 30, np.random.default_rng(3), names=["RX", "RY", "CNOT"])
    cops, tp = capi.Ops(*ops), list(range(sum(1 for p in ops[1] if p)))
    obs = [to_capi(capi, ("named", "PauliZ", [w])) for w in range(3)]
    s = capi.State(n)
    many = [capi.Obs.named("PauliX", [k % n]) for k in range(5000)]
    for o in many:
        s.expval(o)
    del many, o
    capi.adjoint_jacobian(s, obs, cops, tp, True)
    capi.profiling_enable(True)
    try:
        s.expval(capi.Obs.sparse(np.ones(1 << n), np.arange(1 << n), np.arange((1 << n) + 1), list(range(n))))
        assert capi.profiling_get("device_alloc")["launches"] >= 1  # the counter counts: a matrix is allocated
    finally:
        capi.profiling_enable(False)
    capi.profiling_enable(True)
    try:
        for _ in range(3):
            capi.adjoint_jacobian(s, obs, cops, tp, True)
        assert "device_alloc" not in capi.profiling_names() or capi.profiling_get("device_alloc")["launches"] == 0
    finally:
        capi.profiling_enable(False)

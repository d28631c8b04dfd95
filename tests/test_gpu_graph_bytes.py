"""A Jacobian of so many observables that its states alone pass the bound of what
graphs may hold (4 GiB on a device) is launched eagerly and holds nothing after
the call; one of few observables is captured. Both give the same rows, which a
different grouping of the observables changes by roundings of 1e-16 each only."""
import numpy as np
import pytest

from helpers import random_ops

pytestmark = pytest.mark.gpu


def test_graph_larger_than_its_bound(capi):
    n = 19
    rng = np.random.default_rng(19)
    names, params, wires, inv, mats = random_ops(n, 40, rng, names=["RX", "RY", "RZ", "CNOT", "IsingXX"])
    ops = capi.Ops(names, params, wires, inv, mats)
    tps = list(range(sum(1 for p in params if p)))
    s = capi.State(n, np.complex128)  # 8 MiB
    out = {}
    for n_obs in (n, 512):  # 21 states and 514, of which 512 would fit
        obs = [capi.Obs.named("PauliZ", [j % n]) for j in range(n_obs)]
        capi.adjoint_jacobian(s, obs, ops, tps, True)  # a structure's second call captures
        capi.profiling_enable(True)
        try:
            out[n_obs] = capi.adjoint_jacobian(s, obs, ops, tps, True)
            assert ("host_adjoint_graph" in capi.profiling_names()) == (n_obs == n)
        finally:
            capi.profiling_enable(False)
    np.testing.assert_allclose(out[512], out[n][np.arange(512) % n], rtol=0, atol=1e-12)

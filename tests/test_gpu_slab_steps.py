"""Consecutive two-state steps taken in one launch (a workgroup owns the slab
of amplitudes their wires span) against the oracle: states smaller than a slab,
one slab and many, gates that repeat and share wires (each step reads what the
last one wrote), wires at both ends, fixed gates between trainable ones, and more
observables than a launch holds."""
import numpy as np
import pytest

import oracle as O
from helpers import random_state, to_capi, to_oracle

pytestmark = pytest.mark.gpu


def excitations(n, count, rng):
    names, params, wires, inverses = [], [], [], []
    for k in range(count):
        name = ("DoubleExcitation", "SingleExcitation", "DoubleExcitationPlus", "Toffoli")[rng.choice(4, p=[.4, .3, .2, .1])]
        m = {"SingleExcitation": 2, "Toffoli": 3}.get(name, 4)
        w = [int(x) for x in rng.choice(n, m, replace=False)]
        if k % 3 == 2 and len(wires[-1]) == m:
            w = wires[-1][::-1]
        names.append(name)
        params.append([] if name == "Toffoli" else [float(rng.uniform(0, 6))])
        wires.append(w)
        inverses.append(bool(rng.integers(2)))
    return names, params, wires, inverses, [[] for _ in names]


# 1e-10 / 1e-5 for derivatives, 1e-12 / 2e-5 for amplitudes: as the other step tests.
@pytest.mark.parametrize("dtype,jtol,atol", [(np.complex128, 1e-10, 1e-12), (np.complex64, 1e-5, 2e-5)])
@pytest.mark.parametrize("n,n_obs", [(4, 1), (6, 3), (7, 2), (11, 8), (12, 1), (13, 9), (14, 5), (16, 2)])
def test_slab_steps_match_oracle(capi, n, n_obs, dtype, jtol, atol):
    rng = np.random.default_rng(100 * n + n_obs)
    ops = excitations(n, 40, rng)
    psi = random_state(n, rng).astype(dtype)
    obs = [("named", "PauliZ", [j % n]) for j in range(n_obs)]
    npar = sum(1 for p in ops[1] if p)
    tp = sorted(int(t) for t in rng.choice(npar, max(1, 2 * npar // 3), replace=False))
    s = capi.State(n, dtype)
    s.upload(psi)
    ref = O.adjoint_jacobian(psi.astype(np.complex128), [to_oracle(o) for o in obs], O.Ops(*ops), tp, True)
    for _ in range(4):  # launched, captured, replayed
        got = capi.adjoint_jacobian(s, [to_capi(capi, o) for o in obs], capi.Ops(*ops), tp, True)
        np.testing.assert_allclose(got, ref, rtol=0, atol=jtol)
    s.apply_ops(capi.Ops(*ops))
    np.testing.assert_allclose(s.download(), O.apply_ops(psi.astype(np.complex128), O.Ops(*ops)), rtol=0, atol=atol)

"""Op lists with explicit one-wire matrices that are not unitary (scaled,
projectors, zero) among rotations, at sizes of the one-launch and of the
pass-by-pass path, both precisions, against the oracle: amplitudes at 1e-12 and
2e-5 of the state's norm."""
import numpy as np
import pytest

import oracle as O

pytestmark = pytest.mark.gpu

MATRICES = {
    "scaled": [2, 0, 0, 2],
    "projector": [1, 0, 0, 0],
    "plus projector": [0.5, 0.5, 0.5, 0.5],
    "lopsided": [0.5, 0.25j, -0.3, 1.5],
    "zero": [0, 0, 0, 0],
    "tiny": [1e-60, 0, 0, 1e-60],
}


def scaled_circuit(n, matrix, rng):
    ops = [("Hadamard", [w], [], []) for w in range(n)]
    for w in range(n):
        ops.append(("RX", [w], [float(rng.uniform(0, 2 * np.pi))], []))
    ops.append(("CNOT", [0, n - 1], [], []))
    ops.append(("Matrix", [0], [], np.asarray(matrix, dtype=np.complex128)))
    for w in range(n):
        for g in ("RY", "RZ"):
            ops.append((g, [w], [float(rng.uniform(0, 2 * np.pi))], []))
    ops.append(("Matrix", [n // 2], [], np.asarray(matrix, dtype=np.complex128)))
    ops += [("CNOT", [w, w + 1], [], []) for w in range(n - 1)]
    ops += [("RX", [w], [float(rng.uniform(0, 2 * np.pi))], []) for w in range(n)]
    return [[o[0] for o in ops], [o[2] for o in ops], [o[1] for o in ops], [False] * len(ops), [o[3] for o in ops]]


@pytest.mark.parametrize("dtype", [np.complex64, np.complex128])
@pytest.mark.parametrize("n", [5, 12, 13, 14])
@pytest.mark.parametrize("kind", sorted(MATRICES))
def test_apply_ops(capi, kind, n, dtype):
    rng = np.random.default_rng(31 * n + len(kind))
    ops = scaled_circuit(n, MATRICES[kind], rng)
    s = capi.State(n, dtype)
    s.apply_ops(capi.Ops(*ops))
    ref = O.apply_ops(O.zero_state(n), O.Ops(*ops))
    tol = (1e-12 if dtype == np.complex128 else 2e-5) * max(np.linalg.norm(ref), 1e-30)
    np.testing.assert_allclose(s.download(), ref, rtol=0, atol=tol)

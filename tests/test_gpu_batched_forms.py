"""Batched circuits with runs of one-wire gates that lose structure where
angles agree: a rotation and its inverse, a rotation on either side of a Pauli
gate, echoes of both. A plan serves every angle of its patched gates, so
distances of 1 to 10 between the two gates of a wire, in the op list of a whole
and of a staged circuit, unequal angles first, then equal ones on the same plan,
against the oracle at the tolerances of the other batched tests."""
import numpy as np
import pytest

import oracle as O
from helpers import to_capi, to_oracle

pytestmark = pytest.mark.gpu

# The gates of a wire: "+" and "-" mark a rotation and an inverse one.
RUNS = {
    "inverse": lambda g: [g + "+", g + "-"],
    "X between": lambda g: [g + "+", "PauliX", g + "+"],
    "Y between": lambda g: [g + "+", "PauliY", g + "+"],
    "Z between": lambda g: [g + "+", "PauliZ", g + "+"],
    "echo": lambda g: [g + "+", "PauliX", g + "+", "PauliX"],
    "S between": lambda g: ["S", g + "+", "PauliZ", g + "-", "Hadamard", "RY+"],
}


def layered(n, gate, kind, gap, rng):
    """The run's gates layer by layer on wires 0 .. gap - 1, so that the gates
    of a wire stand gap ops apart, then CNOTs and a last rotation everywhere."""
    ops = [("Hadamard", [w], []) for w in range(n)]
    for g in RUNS[kind](gate):
        for w in range(gap):
            ops.append((g, [w], [0.0] if g[-1] in "+-" else []))
    ops += [("CNOT", [w, w + 1], []) for w in range(n - 1)]
    ops += [("RX+", [w], [0.0]) for w in range(n)]
    names = [g.rstrip("+-") for g, _, _ in ops]
    return [names, [p for _, _, p in ops], [w for _, w, _ in ops], [g.endswith("-") for g, _, _ in ops],
            [[] for _ in ops]]


@pytest.mark.parametrize("dtype,rtol,atol", [(np.complex128, 1e-10, 1e-12), (np.complex64, 0.0, 1e-5)])
@pytest.mark.parametrize("n,whole", [(10, ""), (13, "10")])
@pytest.mark.parametrize("kind", sorted(RUNS))
def test_run_forms_hold_for_every_angle(capi, monkeypatch, kind, n, whole, dtype, rtol, atol):
    if whole:
        monkeypatch.setenv("PLK_BATCH_WHOLE_QUBITS", whole)
    rng = np.random.default_rng(500 + n)
    circuits = [layered(n, gate, kind, gap, rng) for gate in ("RX", "RY", "RZ") for gap in range(1, 11)]
    obs = ("ham", [0.4, -0.9, 1.3], [("named", "PauliX", [0]), ("named", "PauliY", [n // 2]),
                                     ("tensor", [("named", "PauliZ", [1]), ("named", "PauliX", [2])])])
    for equal in (False, True):
        for ops in circuits:
            value = float(rng.uniform(0, 2 * np.pi))
            ops[1] = [[value if equal else float(rng.uniform(0, 2 * np.pi))] if p else [] for p in ops[1]]
        trainable = [list(range(sum(1 for p in ops[1] if p))) for ops in circuits]
        values, rows = capi.adjoint_batched([n] * len(circuits), [capi.Ops(*ops) for ops in circuits],
                                            [to_capi(capi, obs)] * len(circuits), trainable, dtype=dtype)
        for ops, tp, v, row in zip(circuits, trainable, values, rows):
            o = O.Ops(*ops)
            psi = O.apply_ops(O.zero_state(n), o)
            np.testing.assert_allclose(v, O.expval(psi, to_oracle(obs)), rtol=rtol, atol=atol)
            ref = O.adjoint_jacobian(O.zero_state(n), [to_oracle(obs)], o, tp, True)[0]
            np.testing.assert_allclose(row, ref, rtol=rtol, atol=atol)


@pytest.mark.parametrize("dtype,rtol,atol", [(np.complex128, 1e-10, 1e-12), (np.complex64, 0.0, 1e-5)])
@pytest.mark.parametrize("gate", ["RX", "RY", "RZ", "PhaseShift"])
def test_named_gate_with_matrix(capi, gate, dtype, rtol, atol):
    """A named gate is the gate whatever matrix its op carries, in a run with
    other rotations too; two calls with other angles."""
    n, rng = 4, np.random.default_rng(12)
    names = ["Hadamard", gate, "RZ", "CNOT", "RY", gate]
    wires = [[0], [0], [0], [0, 1], [1], [1]]
    mats = [[], np.array([0, 1, 1, 0], dtype=np.complex128), [], [], [], np.array([1, 0, 0, 2], dtype=np.complex128)]
    obs = ("ham", [0.7, 0.2], [("named", "PauliY", [0]), ("named", "PauliX", [1])])
    for _ in range(2):
        params = [[], [float(rng.uniform(0, 6))], [float(rng.uniform(0, 6))], [], [float(rng.uniform(0, 6))],
                  [float(rng.uniform(0, 6))]]
        ops = (names, params, wires, [False, True, False, False, False, False], mats)
        values, rows = capi.adjoint_batched([n], [capi.Ops(*ops)], [to_capi(capi, obs)], [[0, 1, 2, 3]], dtype=dtype)
        o = O.Ops(*ops)
        np.testing.assert_allclose(values[0], O.expval(O.apply_ops(O.zero_state(n), o), to_oracle(obs)), rtol=rtol,
                                   atol=atol)
        np.testing.assert_allclose(rows[0], O.adjoint_jacobian(O.zero_state(n), [to_oracle(obs)], o, [0, 1, 2, 3], True)[0],
                                   rtol=rtol, atol=atol)

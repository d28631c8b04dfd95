"""What this framework is timed on: the calls that variational, sampling and
simulation programs make, from a five-qubit training step to the 24-qubit
Jacobian and 26-qubit circuits, in both precisions.

A case is a dict of plain values: its kind, its sizes, the precision of the
state and `layout`, the seed of the circuit's structure (gates, wires, Pauli
words). The structure is what a program keeps; angles, coefficients and states
are its inputs and come from the seed given to `prepare`.
"""
import math
import os
import random
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.getcwd(), "pennylane-lightning-kokkos_amd"))

from pennylane_lightning_kokkos_amd import _capi  # noqa: E402
from pennylane_lightning_kokkos_amd.torch_adjoint import Circuit, Op, make_function  # noqa: E402

TWO_PI = 2.0 * math.pi


# ---------------------------------------------------------------------------
# The cases.
# ---------------------------------------------------------------------------
def listed():
    return [
        # The smallest call: one optimiser step of a five-qubit variational
        # circuit through torch (expectation values, then the gradient).
        {"name": "train_5q_f64", "kind": "train", "ansatz": "entangling", "qubits": 5, "layers": 2,
         "words": 8, "observables": 2, "dtype": "complex128", "layout": 1},
        # The small Jacobian: 12 qubits, 144 parameters, PauliZ on each wire.
        {"name": "jacobian_12q_c128", "kind": "jacobian", "ansatz": "rotations", "qubits": 12, "layers": 4,
         "words": 0, "observables": 12, "dtype": "complex128", "layout": 2},
        # An odd-sized Jacobian in single precision, kept in float32.
        {"name": "jacobian_17q_c64", "kind": "jacobian", "ansatz": "entangling", "qubits": 17, "layers": 5,
         "words": 20, "observables": 5, "dtype": "complex64", "layout": 3},
        # A chemistry ansatz: excitations from the Hartree-Fock state.
        {"name": "jacobian_excitations_20q", "kind": "jacobian", "ansatz": "excitations", "qubits": 20,
         "layers": 60, "words": 32, "observables": 5, "dtype": "complex128", "layout": 4},
        # The headline: 24 qubits, 720 parameters, 8 PauliZ and a Hamiltonian.
        {"name": "jacobian_24q_c128", "kind": "jacobian", "ansatz": "entangling", "qubits": 24, "layers": 10,
         "words": 32, "observables": 9, "dtype": "complex128", "layout": 5},
        # A training step in single precision: one expectation value forward,
        # its gradient backward.
        {"name": "train_22q_f32", "kind": "train", "ansatz": "entangling", "qubits": 22, "layers": 4,
         "words": 22, "observables": 1, "dtype": "complex64", "layout": 6},
        # Forward simulation: a random gate stream on a 1 GiB state.
        {"name": "stream_26q_c128", "kind": "stream", "qubits": 26, "gates": 600, "dtype": "complex128", "layout": 7},
        # Random SU(2) layers and CZ bricks as fused five-qubit blocks.
        {"name": "blocks_27q_c64", "kind": "blocks", "qubits": 27, "layers": 6, "dtype": "complex64", "layout": 8},
        # Energy of a 64-word Hamiltonian on a 1 GiB state.
        {"name": "expval_26q_c128", "kind": "expval", "qubits": 26, "words": 64, "dtype": "complex128", "layout": 9},
        # Energy of a sparse Hamiltonian (CSR matrix kept by the program).
        {"name": "csr_19q_c128", "kind": "csr", "qubits": 19, "words": 32, "dtype": "complex128", "layout": 10},
        # Many small circuits of uneven size in one call, kept in float32.
        {"name": "batch_1024_c64", "kind": "batch", "circuits": 1024, "least": 6, "most": 16, "layers": 8,
         "dtype": "complex64", "layout": 11},
        # Reading a state out: marginal probabilities and shots.
        {"name": "measure_23q_c128", "kind": "measure", "qubits": 23, "wires": 9, "shots": 2000,
         "dtype": "complex128", "layout": 12},
    ]


def _log_int(rng, lo, hi):
    return min(hi, max(lo, round(math.exp(rng.uniform(math.log(lo), math.log(hi))))))


def draw(rng):
    kind = rng.choice(["train", "train", "jacobian", "jacobian", "jacobian", "stream", "blocks", "expval", "csr",
                       "batch", "measure"])
    case = {"kind": kind, "dtype": rng.choice(["complex64", "complex128"]), "layout": rng.randrange(1 << 20)}
    if kind in ("train", "jacobian"):
        ansatz = rng.choice(["entangling", "entangling", "rotations", "excitations"])
        excitations = ansatz == "excitations"
        case["ansatz"] = ansatz
        case["qubits"] = rng.randint(6 if excitations else 4, 20 if excitations else 23)
        case["layers"] = _log_int(rng, 5, 60) if excitations else rng.randint(1, 6)
        case["words"] = _log_int(rng, 1, 32)
        case["observables"] = rng.randint(1, 3) if kind == "train" else rng.randint(1, min(9, case["qubits"]))
    elif kind == "stream":
        case.update(qubits=rng.randint(8, 26), gates=_log_int(rng, 20, 600))
    elif kind == "blocks":
        case.update(qubits=rng.randint(9, 27 if case["dtype"] == "complex64" else 26), layers=rng.randint(1, 6))
    elif kind == "expval":
        case.update(qubits=rng.randint(6, 26), words=_log_int(rng, 1, 64))
    elif kind == "csr":
        case.update(qubits=rng.randint(6, 19), words=_log_int(rng, 2, 32))
    elif kind == "batch":
        least = rng.randint(4, 10)
        case.update(circuits=_log_int(rng, 8, 1024), least=least, most=rng.randint(least, 16), layers=rng.randint(1, 8))
    else:
        qubits = rng.randint(6, 25)
        case.update(qubits=qubits, wires=rng.randint(1, min(qubits, 20)), shots=_log_int(rng, 1, 10000))
    return case


# ---------------------------------------------------------------------------
# Structures: gates as (name, wires), Pauli words as {wire: "X" | "Y" | "Z"}.
# ---------------------------------------------------------------------------
ROTATIONS = ("RX", "RY", "RZ", "CRX", "IsingXX", "IsingZZ", "SingleExcitation", "DoubleExcitation")


def circuit_gates(ansatz, n, layers, rng):
    """The gates of a variational circuit and its starting basis state."""
    gates, index = [], 0
    if ansatz == "rotations":  # RX, RY, RZ on every wire, then a CNOT ring
        for _ in range(layers):
            gates += [(g, (w,)) for g in ("RX", "RY", "RZ") for w in range(n)]
            gates += [("CNOT", (w, (w + 1) % n)) for w in range(n)]
    elif ansatz == "entangling":  # Rot on every wire, then CNOTs of growing range
        for layer in range(layers):
            gates += [(g, (w,)) for w in range(n) for g in ("RZ", "RY", "RZ")]
            reach = layer % (n - 1) + 1
            gates += [("CNOT", (w, (w + reach) % n)) for w in range(n)]
    else:  # two DoubleExcitations and one SingleExcitation a layer
        half = n // 2
        index = ((1 << half) - 1) << (n - half)  # the first half of the wires occupied
        for _ in range(layers):
            for _double in range(2):
                gates.append(("DoubleExcitation", tuple(rng.sample(range(half), 2) + rng.sample(range(half, n), 2))))
            gates.append(("SingleExcitation", (rng.randrange(half), rng.randrange(half, n))))
    return gates, index


def stream_gates(n, count, rng):
    pool = ["Hadamard", "RX", "RY", "RZ", "CNOT", "CZ", "CRX", "SWAP", "IsingXX", "IsingZZ"]
    out = []
    for _ in range(count):
        name = rng.choice(pool)
        out.append((name, tuple(rng.sample(range(n), 1 if name in ("Hadamard", "RX", "RY", "RZ") else 2))))
    return out


def pauli_words(n, count, rng):
    out = []
    for _ in range(count):
        wires = sorted(rng.sample(range(n), rng.randint(1, min(4, n))))
        out.append({w: rng.choice("XYZ") for w in wires})
    return out


def observable_words(case, rng):
    """Words of each observable: a Hamiltonian (when there are words), then
    PauliZ on the first wires."""
    n = case["qubits"]
    obs = [pauli_words(n, case["words"], rng)] if case["words"] else []
    return obs + [[{w % n: "Z"}] for w in range(case["observables"] - len(obs))]


def structure(case):
    rng = random.Random(case["layout"])
    kind = case["kind"]
    if kind in ("train", "jacobian"):
        gates, index = circuit_gates(case["ansatz"], case["qubits"], case["layers"], rng)
        return {"gates": gates, "index": index, "obs": observable_words(case, rng)}
    if kind == "stream":
        return {"gates": stream_gates(case["qubits"], case["gates"], rng)}
    if kind == "blocks":
        n, gates = case["qubits"], []
        for layer in range(case["layers"]):
            gates += [("QubitUnitary", (w,)) for w in range(n)]
            gates += [("CZ", (w, w + 1)) for w in range(layer % 2, n - 1, 2)]
        return {"gates": gates}
    if kind in ("expval", "csr"):
        return {"words": pauli_words(case["qubits"], case["words"], rng)}
    if kind == "batch":
        return {"sizes": [(rng.randint(case["least"], case["most"]), rng.randint(1, case["layers"]))
                          for _ in range(case["circuits"])]}
    return {"wires": sorted(rng.sample(range(case["qubits"]), case["wires"]))}


def batch_gates(n, layers):
    """RY and RZ on every wire, then a CNOT chain, `layers` times."""
    gates = []
    for _ in range(layers):
        gates += [(g, (w,)) for g in ("RY", "RZ") for w in range(n)]
        gates += [("CNOT", (w, w + 1)) for w in range(n - 1)]
    return gates


def n_params(gates):
    return sum(1 for name, _ in gates if name in ROTATIONS)


# ---------------------------------------------------------------------------
# Inputs: everything that depends on the seed, in numpy and torch.
# ---------------------------------------------------------------------------
def _angles(gates, rng):
    return rng.uniform(0.0, TWO_PI, size=n_params(gates))


def _haar(rng):
    q, r = np.linalg.qr(rng.normal(size=(2, 2)) + 1j * rng.normal(size=(2, 2)))
    d = np.diag(r)
    q = q * (d / np.abs(d))
    return q / np.sqrt(np.linalg.det(q))


def _device():
    return torch.device("cuda" if torch.cuda.is_available() else "cpu")


def _amplitudes(n, seed, dtype):
    """A normalised state with Gaussian amplitudes, as a deep circuit gives."""
    gen = torch.Generator(device=_device()).manual_seed(seed)
    real = torch.float64 if dtype == "complex128" else torch.float32
    v = torch.view_as_complex(torch.randn(1 << n, 2, generator=gen, device=_device(), dtype=real))
    return v.div_(torch.linalg.vector_norm(v))


def inputs(case, seed):
    s = structure(case)
    rng = np.random.default_rng(seed)
    kind = case["kind"]
    if kind in ("train", "jacobian"):
        s["angles"] = _angles(s["gates"], rng)
        s["coeffs"] = [rng.normal(size=len(words)) if len(words) > 1 else np.ones(len(words)) for words in s["obs"]]
        s["weights"] = rng.normal(size=len(s["obs"]))
    elif kind == "stream":
        s["angles"] = _angles(s["gates"], rng)
    elif kind == "blocks":
        s["matrices"] = [_haar(rng) if name == "QubitUnitary" else None for name, _ in s["gates"]]
    elif kind in ("expval", "csr"):
        s["coeffs"] = rng.normal(size=case["words"])
        s["psi"] = _amplitudes(case["qubits"], seed, case["dtype"])
    elif kind == "batch":
        s["angles"] = [_angles(batch_gates(n, d), rng) for n, d in s["sizes"]]
    else:
        s["psi"] = _amplitudes(case["qubits"], seed, case["dtype"])
        s["shot_seed"] = int(rng.integers(1 << 31))
    return s


# ---------------------------------------------------------------------------
# The framework's side.
# ---------------------------------------------------------------------------
class Amplitudes:
    """A state's amplitudes in HBM for torch, without a copy."""

    def __init__(self, state):
        self.state = state  # keeps the memory
        kind = "<c16" if state.dtype == np.complex128 else "<c8"
        self.__cuda_array_interface__ = {"shape": (state.length,), "typestr": kind, "version": 2,
                                         "data": (state.device_ptr(), False)}


def _view(state):
    return torch.as_tensor(Amplitudes(state), device="cuda")


def _state(psi):
    n = psi.numel().bit_length() - 1
    s = _capi.State(n, np.complex128 if psi.dtype == torch.complex128 else np.complex64)
    _view(s).copy_(psi)
    torch.cuda.synchronize()
    return s


def _word(word):
    return ("tensor", [("named", "Pauli" + p, [w]) for w, p in word.items()])


def _describe(words, coeffs):
    """An observable as the package's plain description."""
    if len(words) == 1 and coeffs[0] == 1.0:
        word = words[0]
        if len(word) == 1:
            (w, p), = word.items()
            return ("named", "Pauli" + p, [w])
        return _word(word)
    return ("ham", [float(c) for c in coeffs], [_word(word) for word in words])


def _obs(desc):
    if desc[0] == "named":
        return _capi.Obs.named(desc[1], desc[2])
    if desc[0] == "tensor":
        return _capi.Obs.tensor([_obs(f) for f in desc[1]])
    return _capi.Obs.hamiltonian(desc[1], [_obs(t) for t in desc[2]])


def _ops(gates, angles, matrices=None):
    it = iter(angles)
    params = [[float(next(it))] if name in ROTATIONS else [] for name, _ in gates]
    mats = [[] if m is None else m.reshape(-1) for m in (matrices or [None] * len(gates))]
    return _capi.Ops([g for g, _ in gates], params, [list(w) for _, w in gates], [False] * len(gates), mats)


def _train_ops(case, gates, index):
    """The circuit as a training program writes it: Rot where it means Rot."""
    n = case["qubits"]
    ops = [Op("PauliX", [w]) for w in range(n) if index >> (n - 1 - w) & 1]
    k = 0
    while k < len(gates):
        name, wires = gates[k]
        if case["ansatz"] == "entangling" and name == "RZ":
            ops.append(Op("Rot", list(wires), [0.0, 0.0, 0.0]))
            k += 3
        else:
            ops.append(Op(name, list(wires), [0.0] if name in ROTATIONS else []))
            k += 1
    return ops


def prepare(case, seed):
    s = inputs(case, seed)
    kind, dtype = case["kind"], np.dtype(case["dtype"])
    state = {"kind": kind, "dtype": case["dtype"]}
    if kind == "train":
        real = torch.float64 if case["dtype"] == "complex128" else torch.float32
        obs = [_describe(w, c) for w, c in zip(s["obs"], s["coeffs"])]
        state["circuit"] = Circuit(case["qubits"], _train_ops(case, s["gates"], s["index"]), obs, dtype)
        state["params"] = torch.tensor(s["angles"], dtype=real, device="cuda", requires_grad=True)
        state["weights"] = torch.tensor(s["weights"], dtype=real, device="cuda")
        state["function"] = make_function()
    elif kind == "jacobian":
        state["state"] = _capi.State(case["qubits"], dtype)
        state["state"].set_basis(s["index"])
        state["obs"] = [_obs(_describe(w, c)) for w, c in zip(s["obs"], s["coeffs"])]
        state["ops"] = _ops(s["gates"], s["angles"])
        state["trainable"] = list(range(len(s["angles"])))
    elif kind == "stream":
        state["state"] = _capi.State(case["qubits"], dtype)
        state["ops"] = _ops(s["gates"], s["angles"])
    elif kind == "blocks":
        state["state"] = _capi.State(case["qubits"], dtype)
        state["ops"] = _ops(s["gates"], [], s["matrices"])
    elif kind == "expval":
        state["state"] = _state(s["psi"])
        state["obs"] = _obs(("ham", [float(c) for c in s["coeffs"]], [_word(w) for w in s["words"]]))
    elif kind == "csr":
        state["state"] = _state(s["psi"])
        data, indices, indptr = csr_matrix(case["qubits"], s["words"], s["coeffs"])
        state["obs"] = _capi.Obs.sparse(data, indices, indptr, list(range(case["qubits"])))
    elif kind == "batch":
        state["qubits"] = [n for n, _ in s["sizes"]]
        state["ops"] = [_ops(batch_gates(n, d), a) for (n, d), a in zip(s["sizes"], s["angles"])]
        of_size = {n: _obs(_describe([{w: "Z"} for w in range(n)], [1.0] * n)) for n in set(state["qubits"])}
        state["obs"] = [of_size[n] for n in state["qubits"]]
    else:
        state["state"] = _state(s["psi"])
        state["wires"], state["shots"], state["seed"] = s["wires"], case["shots"], s["shot_seed"]
    return state


def _kept(values, dtype):
    """Results as a program of this precision keeps them."""
    return torch.from_numpy(values).to(torch.float64 if dtype == "complex128" else torch.float32)


def run(state):
    kind = state["kind"]
    if kind == "train":
        values = state["function"].apply(state["params"], state["circuit"])
        grad, = torch.autograd.grad((values * state["weights"]).sum(), state["params"])
        return {"values": values.detach(), "grad": grad}
    if kind == "jacobian":
        jac = _capi.adjoint_jacobian(state["state"], state["obs"], state["ops"], state["trainable"], True)
        return _kept(jac, state["dtype"])
    if kind == "stream":
        state["state"].reset()
        state["state"].apply_ops(state["ops"])
        return _view(state["state"])
    if kind == "blocks":
        state["state"].reset()
        state["state"].apply_ops_blocks(state["ops"])
        return _view(state["state"])
    if kind in ("expval", "csr"):
        return state["state"].expval(state["obs"])
    if kind == "batch":
        values, rows = _capi.adjoint_batched(state["qubits"], state["ops"], state["obs"], dtype=np.dtype(state["dtype"]))
        return {"values": _kept(values, state["dtype"]), "grad": _kept(np.concatenate(rows), state["dtype"])}
    return {"probs": state["state"].probs(state["wires"]),
            "samples": state["state"].generate_samples(state["shots"], state["seed"])}


def csr_matrix(n, words, coeffs):
    """CSR (data, indices, indptr) of sum_k c_k P_k, columns sorted, one entry
    per row and distinct X mask, built with torch."""
    dev = _device()
    rows = torch.arange(1 << n, device=dev)
    by_mask = {}
    for word, c in zip(words, coeffs):
        flip = sum(1 << (n - 1 - w) for w, p in word.items() if p in "XY")
        sign = sum(1 << (n - 1 - w) for w, p in word.items() if p in "ZY")
        odd = torch.zeros_like(rows)
        for b in range(n):
            if sign >> b & 1:
                odd ^= (rows ^ flip) >> b & 1
        # Y = i X Z on one wire, so a word is i^(number of Y) X^flip Z^sign.
        phase = complex(c) * 1j ** sum(p == "Y" for p in word.values())
        by_mask[flip] = by_mask.get(flip, 0) + phase * (1 - 2 * odd).to(torch.complex128)
    masks = sorted(by_mask)
    cols = torch.stack([rows ^ m for m in masks], dim=1)
    vals = torch.stack([by_mask[m] for m in masks], dim=1)
    cols, order = torch.sort(cols, dim=1)
    vals = torch.gather(vals, 1, order)
    indptr = np.arange(0, (len(masks) << n) + 1, len(masks), dtype=np.int32)
    return vals.reshape(-1).cpu().numpy(), cols.reshape(-1).to(torch.int32).cpu().numpy(), indptr


# ---------------------------------------------------------------------------
# What a pass cannot do without.
# ---------------------------------------------------------------------------
# Flops per amplitude of one gate, by what its matrix leaves to compute.
GATE_FLOPS = {"Hadamard": 4, "RX": 6, "RY": 6, "RZ": 6, "CNOT": 0, "CZ": 0, "SWAP": 0, "CRX": 3, "IsingXX": 6,
              "IsingZZ": 6, "QubitUnitary": 14, "SingleExcitation": 3, "DoubleExcitation": 0.75}


def _sweep_flops(gates, amps, n_obs, words):
    """Forward pass, observables, reverse pass with the inner products."""
    apply = sum(GATE_FLOPS[name] for name, _ in gates) * amps
    return apply * (2 + n_obs) + 8.0 * words * amps + 4.0 * n_obs * n_params(gates) * amps


def work(case):
    s = structure(case)
    kind = case["kind"]
    size = 16 if case["dtype"] == "complex128" else 8
    if kind == "batch":
        flops = bytes_ = 0.0
        for n, d in s["sizes"]:
            gates = batch_gates(n, d)
            flops += _sweep_flops(gates, float(1 << n), 1, n)
            bytes_ += 8.0 * (2 * n_params(gates) + 1)
        return {"bytes": bytes_, "flops": flops}
    amps = float(1 << case["qubits"])
    if kind == "train":
        words = sum(len(w) for w in s["obs"])
        apply = sum(GATE_FLOPS[name] for name, _ in s["gates"]) * amps
        flops = _sweep_flops(s["gates"], amps, 1, words) + apply + 8.0 * words * amps
        return {"bytes": size * amps + 16.0 * n_params(s["gates"]), "flops": flops}
    if kind == "jacobian":
        words = sum(len(w) for w in s["obs"])
        return {"bytes": size * amps + 8.0 * n_params(s["gates"]) * (1 + len(s["obs"])),
                "flops": _sweep_flops(s["gates"], amps, len(s["obs"]), words)}
    if kind in ("stream", "blocks"):
        return {"bytes": 2.0 * size * amps, "flops": sum(GATE_FLOPS[name] for name, _ in s["gates"]) * amps}
    if kind == "expval":
        return {"bytes": size * amps, "flops": 8.0 * amps * case["words"]}
    if kind == "csr":
        masks = len({tuple(w for w, p in word.items() if p in "XY") for word in s["words"]})
        return {"bytes": size * amps + masks * amps * (size + 4) + 4 * (amps + 1), "flops": 8.0 * amps * masks}
    return {"bytes": size * amps + 8.0 * (1 << case["wires"]) + 8.0 * case["shots"] * case["qubits"],
            "flops": 4.0 * amps}


# ---------------------------------------------------------------------------
# The same results in 64 bits by plain torch: gates as matrices applied to
# strided slices of a batch of states, gradients by the reverse walk.
# ---------------------------------------------------------------------------
PAULI = {"X": [[0, 1], [1, 0]], "Y": [[0, -1j], [1j, 0]], "Z": [[1, 0], [0, -1]]}
SWAP = [[1, 0, 0, 0], [0, 0, 1, 0], [0, 1, 0, 0], [0, 0, 0, 1]]


def _kron(a, b):
    k = len(b)
    return [[a[r // k][c // k] * b[r % k][c % k] for c in range(len(a) * k)] for r in range(len(a) * k)]


def _eye(d):
    return [[1 if r == c else 0 for c in range(d)] for r in range(d)]


def _rotation(generator, t):
    """exp(-i t/2 G) for G^2 = 1 on the states that G moves: t is a number or
    one angle per state of the batch."""
    if isinstance(t, torch.Tensor):
        c, s = torch.cos(t / 2).to(torch.complex128), torch.sin(t / 2).to(torch.complex128)
    else:
        c, s = math.cos(t / 2), math.sin(t / 2)
    d = len(generator)
    out = _eye(d)
    for r in range(d):
        if any(generator[r]):
            out[r] = [(c if r == k else 0) + (-1j * s * generator[r][k] if generator[r][k] != 0 else 0)
                      for k in range(d)]
    return out


def _generator(name):
    if name in ("RX", "RY", "RZ"):
        return PAULI[name[1]]
    if name == "CRX":
        return _kron([[0, 0], [0, 1]], PAULI["X"])
    if name in ("IsingXX", "IsingZZ"):
        return _kron(PAULI[name[-1]], PAULI[name[-1]])
    d, lo = (4, 1) if name == "SingleExcitation" else (16, 3)
    g = [[0] * d for _ in range(d)]
    g[lo][d - 1 - lo], g[d - 1 - lo][lo] = -1j, 1j
    return g


def _matrix(name, t=None):
    if name in ROTATIONS:
        return _rotation(_generator(name), t)
    if name == "Hadamard":
        h = math.sqrt(0.5)
        return [[h, h], [h, -h]]
    if name == "CNOT":
        return [[1, 0, 0, 0], [0, 1, 0, 0], [0, 0, 0, 1], [0, 0, 1, 0]]
    if name == "CZ":
        return [[1, 0, 0, 0], [0, 1, 0, 0], [0, 0, 1, 0], [0, 0, 0, -1]]
    return SWAP


def _is(x, value):
    return not isinstance(x, torch.Tensor) and x == value


def _apply(v, n, wires, m):
    """m on `wires` of every state of v (batch, 2^n); entries are numbers or
    one value per state of the batch."""
    order = sorted(wires)
    shape, last = [v.shape[0]], -1
    for w in order:
        shape += [1 << (w - last - 1), 2]
        last = w
    shape.append(1 << (n - 1 - last))
    x = v.reshape(shape)
    out = torch.empty_like(x)
    k = len(wires)

    def at(local):
        bit = {w: local >> (k - 1 - j) & 1 for j, w in enumerate(wires)}
        index = [slice(None)]
        for w in order:
            index += [slice(None), bit[w]]
        return tuple(index)

    def scaled(c, value):
        part = x[at(c)]
        return part * (value.reshape([-1] + [1] * (part.dim() - 1)) if isinstance(value, torch.Tensor) else value)

    for r in range(1 << k):
        row = [c for c in range(1 << k) if not _is(m[r][c], 0)]
        if row == [r] and _is(m[r][r], 1):
            out[at(r)] = x[at(r)]
            continue
        acc = None
        for c in row:
            term = scaled(c, m[r][c])
            acc = term if acc is None else acc.add_(term)
        out[at(r)] = 0 if acc is None else acc
    return out.reshape(v.shape)


def _dagger(m):
    conj = (lambda e: e.conj() if isinstance(e, torch.Tensor) else complex(e).conjugate() if e not in (0, 1) else e)
    return [[conj(m[c][r]) for c in range(len(m))] for r in range(len(m))]


def _observe(v, n, words, coeffs):
    out = torch.zeros_like(v)
    for word, c in zip(words, coeffs):
        t = v
        for w, p in word.items():
            t = _apply(t, n, (w,), PAULI[p])
        out.add_(t, alpha=float(c))
    return out


def _overlap(a, b):
    """<a|b> per row, in the batch's rows."""
    return torch.linalg.vecdot(a, b, dim=-1)


def _sweep(n, gates, angles, index, obs, coeffs, batch=1):
    """Expectation values and Jacobian of `batch` circuits of one structure;
    angles[k] is the k-th parameter, a number or one per circuit."""
    phi = torch.zeros(batch, 1 << n, dtype=torch.complex128, device=_device())
    phi[:, index] = 1
    it = iter(angles)
    mats = [_matrix(name, next(it) if name in ROTATIONS else None) for name, _ in gates]
    for (_, wires), m in zip(gates, mats):
        phi = _apply(phi, n, wires, m)
    hs = [_observe(phi, n, words, c) for words, c in zip(obs, coeffs)]
    values = torch.stack([_overlap(phi, h).real for h in hs])
    jac = torch.zeros(len(obs), n_params(gates), batch, dtype=torch.float64, device=_device())
    k = n_params(gates)
    for (name, wires), m in zip(reversed(gates), reversed(mats)):
        if name in ROTATIONS:
            k -= 1
            g = _apply(phi, n, wires, _generator(name))
            for j, h in enumerate(hs):
                jac[j, k] = _overlap(h, g).imag
        back = _dagger(m)
        phi = _apply(phi, n, wires, back)
        hs = [_apply(h, n, wires, back) for h in hs]
    return values, jac


def exact(case, seed):
    s = inputs(case, seed)
    kind, n = case["kind"], case.get("qubits")
    if kind in ("train", "jacobian"):
        angles = s["angles"]
        if kind == "train" and case["dtype"] == "complex64":
            angles = angles.astype(np.float32).astype(np.float64)  # parameters are held in float32
        values, jac = _sweep(n, s["gates"], [float(a) for a in angles], s["index"], s["obs"], s["coeffs"])
        if kind == "jacobian":
            return jac[:, :, 0]
        real = torch.float64 if case["dtype"] == "complex128" else torch.float32
        weights = torch.tensor(s["weights"], dtype=real).to(jac)
        return {"values": values[:, 0], "grad": weights @ jac[:, :, 0]}
    if kind in ("stream", "blocks"):
        psi = torch.zeros(1, 1 << n, dtype=torch.complex128, device=_device())
        psi[0, 0] = 1
        it = iter(s.get("angles", ()))
        for k, (name, wires) in enumerate(s["gates"]):
            if name == "QubitUnitary":
                m = [[complex(e) for e in row] for row in s["matrices"][k]]
            else:
                m = _matrix(name, float(next(it)) if name in ROTATIONS else None)
            psi = _apply(psi, n, wires, m)
        return psi[0]
    if kind in ("expval", "csr"):
        psi = s["psi"].to(torch.complex128).reshape(1, -1)
        return float(sum(c * _overlap(psi, _observe(psi, n, [w], [1.0])).real
                         for w, c in zip(s["words"], s["coeffs"])))
    if kind == "batch":
        values, grads = [None] * len(s["sizes"]), [None] * len(s["sizes"])
        for size in sorted(set(s["sizes"])):
            q, depth = size
            which = [k for k, x in enumerate(s["sizes"]) if x == size]
            angles = torch.tensor(np.stack([s["angles"][k] for k in which], axis=1), device=_device())
            e, jac = _sweep(q, batch_gates(q, depth), list(angles), 0, [[{w: "Z"} for w in range(q)]], [np.ones(q)],
                            batch=len(which))
            for column, k in enumerate(which):
                values[k], grads[k] = e[0, column], jac[0, :, column]
        return {"values": torch.stack(values), "grad": torch.cat(grads)}
    p = s["psi"].to(torch.complex128).abs().square()
    for w in reversed(range(n)):  # unmeasured wires, the fastest first
        if w not in s["wires"]:
            after = sum(1 for x in s["wires"] if x > w)
            p = p.reshape(-1, 2, 1 << after).sum(dim=1)
    return {"probs": p.reshape(-1), "samples": None}

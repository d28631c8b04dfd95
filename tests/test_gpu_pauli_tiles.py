"""Expectation values of many-word Pauli sums through tiles in LDS: states at
and above the dispatch line, X masks on the lowest and highest bits, several
words with one mask and different Y counts, diagonal words, and words wider
than a tile (which keep the gathers). Against the gather kernel through the
allocation-free entry point and, at the smallest size, the oracle, at 1e-12 of
the sum of the coefficients' sizes (FP64 sums in another order)."""
import numpy as np
import pytest

import oracle as O
from helpers import random_hamiltonian, random_state, to_capi, to_oracle

pytestmark = pytest.mark.gpu


def word(letters):
    return ("tensor", [("named", "Pauli" + p, [w]) for w, p in sorted(letters.items())])


def hamiltonian(n, kind, rng):
    if kind == "random":
        return random_hamiltonian(n, 40, rng)
    if kind == "shared":  # one mask, real and imaginary words, signs on every bit
        letters = []
        for k in range(24):
            x = sorted(int(w) for w in rng.choice(n, 3, replace=False)) if k % 3 == 0 else x
            l = {w: "XY"[int(rng.integers(2))] for w in x}
            for w in rng.choice(n, 4, replace=False):
                l.setdefault(int(w), "Z")
            letters.append(l)
    elif kind == "edges":  # the lowest and highest index bits, and diagonal words
        letters = [{n - 1: "X"}, {n - 2: "Y"}, {n - 3: "X", 0: "Y"}, {0: "X"}, {1: "Y"}, {0: "X", 1: "X"},
                   {n - 1: "Y", n - 2: "Y"}, {0: "Z", n - 1: "Z"}, {3: "Z"}, {5: "X"}, {6: "Y"}, {7: "X", 8: "X"},
                   {9: "X"}, {10: "X"}, {11: "Y"}, {4: "X"}]
    else:  # a word on more wires than a tile has free bits
        letters = [{w: "X" for w in range(14)}] + [{w: "X"} for w in range(8)]
    return ("ham", [float(c) for c in rng.normal(size=len(letters))], [word(l) for l in letters])


@pytest.mark.parametrize("dtype", [np.complex128, np.complex64])
@pytest.mark.parametrize("n", [19, 20, 21, 23])
@pytest.mark.parametrize("kind", ["random", "shared", "edges", "wide"])
def test_tiles_match_gathers(n, kind, dtype):
    from pennylane_lightning_kokkos_amd import _capi

    rng = np.random.default_rng(n)
    ham = hamiltonian(n, kind, rng)
    psi = random_state(n, rng).astype(dtype)
    s = _capi.State(n, dtype)
    s.upload(psi)
    ob = to_capi(_capi, ham)
    tol = 1e-12 * sum(abs(c) for c in ham[1])
    got = s.expval(ob)
    assert abs(got - s.expval_noalloc(ob)) < tol
    assert got == s.expval(ob)
    if n == 20:
        v = psi.astype(np.complex128)
        ref = np.vdot(v, O.obs_apply(v.copy(), to_oracle(ham))).real  # obs_apply works in place
        assert abs(got - ref) < 10 * tol

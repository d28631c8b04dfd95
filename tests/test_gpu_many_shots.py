"""Many shots of a state of at most 4096 amplitudes (a thread a shot) against the
oracle, on both sides of the number of shots from which that is so, at the edges
of a run (64 amplitudes) and with runs without weight; and a basis state."""
import numpy as np
import pytest

import oracle as O
from helpers import random_state, sample_uniforms

pytestmark = pytest.mark.gpu


def _indices(rows):
    n = rows.shape[1]
    return (rows.astype(np.int64) << np.arange(n - 1, -1, -1)).sum(axis=1)


@pytest.mark.parametrize("dtype", [np.complex128, np.complex64])
@pytest.mark.parametrize("n", [1, 2, 5, 6, 7, 8, 11, 12, 13])
def test_many_shots(capi, n, dtype):
    psi = random_state(n, np.random.default_rng(40 + n))
    if n >= 7:
        psi[: 2 ** n // 3] = 0
        psi[-(2 ** n // 5):] = 0
        psi /= np.linalg.norm(psi)
    s = capi.State(n, dtype)
    s.upload(psi.astype(dtype))
    psi = s.download().astype(np.complex128)
    for shots, seed in ((8191, 3), (8192, 5), (16384, 7), (70001, 11)):
        got = _indices(s.generate_samples(shots, seed))
        np.testing.assert_array_equal(got, O.sample_indices(psi, sample_uniforms(seed, shots)))


@pytest.mark.parametrize("n,index", [(1, 1), (6, 63), (12, 64), (12, 4095), (9, 0)])
def test_basis_state(capi, n, index):
    s = capi.State(n, np.complex128)
    s.set_basis(index)
    assert (_indices(s.generate_samples(40000, 1)) == index).all()

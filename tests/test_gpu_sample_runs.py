"""Sampling through run and chunk totals, and marginals whose lowest measured
bits are summed together, against the oracle (MeasuresKokkos.hpp:389-569) at
the edges of a run (64 amplitudes), of a chunk (4096) and of the chunk search's
first level (64 chunks)."""
import numpy as np
import pytest

import oracle as O
from helpers import random_state, sample_uniforms

pytestmark = pytest.mark.gpu


def _indices(rows):
    n = rows.shape[1]
    return (rows.astype(np.int64) << np.arange(n - 1, -1, -1)).sum(axis=1)


@pytest.mark.parametrize("dtype", [np.complex128, np.complex64])
@pytest.mark.parametrize("n", [1, 5, 6, 7, 11, 12, 13, 18, 19, 21])
def test_samples_at_run_and_chunk_edges(capi, n, dtype):
    psi = random_state(n, np.random.default_rng(n))
    if n >= 7:
        psi[: 2 ** n // 3] = 0  # leading runs without weight
        psi[-(2 ** n // 5):] = 0  # and trailing ones
        psi /= np.linalg.norm(psi)
    s = capi.State(n, dtype)
    s.upload(psi.astype(dtype))
    psi = s.download().astype(np.complex128)
    # The largest uniforms may exceed a complex64 state's total (its norm is 1
    # to rounding): the last bin then, as in the oracle.
    for shots, seed in ((1, 3), (3, 5), (700, 11)):
        got = _indices(s.generate_samples(shots, seed))
        np.testing.assert_array_equal(got, O.sample_indices(psi, sample_uniforms(seed, shots)))


@pytest.mark.parametrize("n,index", [(1, 1), (6, 63), (12, 64), (13, 4096), (13, 8191), (20, 2 ** 19 + 4095)])
def test_samples_of_a_basis_state(capi, n, index):
    psi = np.zeros(2 ** n, np.complex128)
    psi[index] = 1
    s = capi.State(n, np.complex128)
    s.upload(psi)
    assert (_indices(s.generate_samples(500, 1)) == index).all()


# 1e-12: sums of at most 2^18 products of FP64 rounding 1e-16 each, of total 1.
@pytest.mark.parametrize("dtype", [np.complex128, np.complex64])
@pytest.mark.parametrize("n", [7, 8, 12, 18])
def test_marginals_with_low_wires(capi, n, dtype):
    s = capi.State(n, dtype)
    s.upload(random_state(n, np.random.default_rng(90 + n)).astype(dtype))
    psi = s.download().astype(np.complex128)
    low = [n - 1, n - 2, n - 3, n - 4, n - 5]
    for wires in ([], low[:1], low[:2], low[:3], low[:4], low[:5], low[::-1], [low[1], 0, low[0]],
                  [0, low[2]], [low[3], low[0], 1, low[2]], [2, 0, 1]):
        got = s.probs(wires) if wires else s.probs([n // 2])
        ref = O.probs(psi, wires if wires else [n // 2])
        np.testing.assert_allclose(got, ref, rtol=0, atol=1e-12, err_msg=f"{wires}")

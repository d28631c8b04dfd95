"""Two fused 5-qubit blocks in one pass (matrix cores, tile in LDS) against the
operations applied one by one: block bits disjoint, shared, at both ends
of the register, and an odd number of blocks."""
import numpy as np
import pytest

from helpers import random_state, random_unitary

pytestmark = pytest.mark.gpu

WIRES = {
    "disjoint": [[0, 4, 8, 12, 16], [2, 6, 10, 14, 18]],
    "low": [[16, 17, 18, 19, 20], [11, 12, 13, 14, 15]],
    "high": [[0, 1, 2, 3, 4], [5, 6, 7, 8, 9]],
    "ends": [[0, 1, 2, 3, 4], [20, 19, 18, 17, 16]],
    "shared": [[3, 20, 7, 11, 5], [20, 7, 0, 1, 19]],
    "four shared": [[1, 9, 13, 17, 18], [18, 17, 13, 9, 2]],
    "odd": [[18, 3, 9, 1, 12], [0, 20, 10, 5, 15], [19, 2, 18, 7, 4]],
}


# complex64: 2e-5 an amplitude, the bar of every complex64 block; complex128: 1e-12.
@pytest.mark.parametrize("dtype,tol", [(np.complex64, 2e-5), (np.complex128, 1e-12)])
@pytest.mark.parametrize("kind", sorted(WIRES))
@pytest.mark.parametrize("n", [21, 22])
def test_pairs_match_single_operations(capi, n, kind, dtype, tol):
    rng = np.random.default_rng(len(kind) + n)
    blocks = WIRES[kind]
    mats = [random_unitary(32, rng) for _ in blocks]
    psi = random_state(n, rng)
    s = capi.State(n, dtype)
    s.upload(psi.astype(dtype))
    assert s.apply_ops_blocks(capi.Ops(["QubitUnitary"] * len(blocks), [[]] * len(blocks), blocks,
                                       [False] * len(blocks), [m.reshape(-1) for m in mats])) == len(blocks)
    ref = capi.State(n, np.complex128)
    ref.upload(psi)
    for b, m in zip(blocks, mats):
        ref.apply_matrix(m, b, False)
    np.testing.assert_allclose(s.download(), ref.download(), atol=tol)

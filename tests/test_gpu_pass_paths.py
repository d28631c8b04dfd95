"""The pass-by-pass paths at sizes that run whole in one launch by default: the
graph tests and the register-tile tests of at most 12 qubits once more with
PLK_SWEEP=0, each checked, by the names the profile holds, to have taken the
path it is about; and batches in which whole and staged circuits mix.

(Circuits of at most 12 qubits with Pauli observables run in one launch before
any graph is captured or pass launched; graphs serve 13 to 21 qubits, and
PLK_BATCH_WHOLE_QUBITS is the widest circuit of a batch that runs whole.)"""
import numpy as np
import pytest

from test_gpu_batched import _check, _random_batch
from test_gpu_graph import (test_graph_c1_workload, test_graph_input_state_changes,  # noqa: F401
                            test_graph_layout_change_recaptures, test_graph_many_structures,
                            test_graph_replays_match_eager_and_oracle)
from test_gpu_rtile import (rtile, test_rtile_adjoint_layered, test_rtile_adjoint_random,  # noqa: F401
                            test_rtile_forward, test_side_by_side_chunks)

pytestmark = pytest.mark.gpu


@pytest.fixture(autouse=True)
def taken_path(request, capi, monkeypatch):
    if "batched" in request.node.name:
        yield
        return
    name = request.node.originalname
    monkeypatch.setenv("PLK_SWEEP", "0")
    monkeypatch.setenv("PLK_GRAPH", "1" if "graph" in name else "0")
    capi.profiling_enable(True)
    yield
    names = capi.profiling_names()
    capi.profiling_enable(False)
    assert "circuit_sweep" not in names
    assert ("host_adjoint_graph" if "graph" in name else "apply_rtile" if "forward" in name else "adjoint_rtile") in names


@pytest.mark.parametrize("dtype", [np.complex128, np.complex64])
@pytest.mark.parametrize("whole", [9, 10, 11])
def test_batched_whole_and_staged(capi, monkeypatch, dtype, whole):
    monkeypatch.setenv("PLK_BATCH_WHOLE_QUBITS", str(whole))
    rng = np.random.default_rng(172 + whole)
    circuits, tps = _random_batch(rng, 24, 3, 13, nops=40)
    assert any(n > 11 for n, _, _ in circuits) and any(n <= 9 for n, _, _ in circuits)
    _check(capi, circuits, tps, dtype)

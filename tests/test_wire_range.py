"""Wires that a size_t does not hold, and bare numbers in place of an op's wire
list, are refused where handles are made, before any device call."""
import numpy as np
import pytest

from pennylane_lightning_kokkos_amd import _capi


@pytest.mark.parametrize("wire", [2**64, 2**64 + 1, 2**80, -1, -2**70])
@pytest.mark.parametrize("form", [list, tuple])
def test_wire_out_of_range(wire, form):
    with pytest.raises(OverflowError):
        _capi.Obs.named("PauliZ", form([wire]))
    with pytest.raises(OverflowError):
        _capi.Ops(["CNOT"], [[]], [form([0, wire])], [False])


def test_wire_forms():
    for wires in ([1], (1,), np.array([1]), [np.int32(1)], [True], range(1, 2), [2**64 - 1]):
        _capi.Obs.named("PauliZ", wires)
        assert _capi.Ops(["RX"], [[0.1]], [wires], [False])._num_par == 1


@pytest.mark.parametrize("wires", [3, 1.5, np.array(3), np.float64(3.0)])
def test_wires_are_a_list(wires):
    with pytest.raises(TypeError):
        _capi.Ops(["RX"], [[0.1]], [wires], [False])

"""ParamCircuit.circ is an attribute that can be assigned, and only the rotations have
parameterised tensors."""

import numpy as np
import pytest

from qxhip import circuits, gradients


def test_circ_can_be_assigned():
    pc = object.__new__(gradients.ParamCircuit)      # (no device)
    pc._circ, pc._angles = circuits.create_param_rqc_circuit(2, 2, 2, seed=1), np.zeros(0)
    other = circuits.create_param_rqc_circuit(2, 2, 2, seed=2)
    pc.circ = other
    assert pc.circ is other and np.array_equal(pc.params(), other.params())
    moved = other.params() + 0.25
    pc._angles = moved
    assert np.array_equal(pc.params(), moved)


@pytest.mark.parametrize("deriv", [False, True])
def test_other_gates_have_no_parameterised_tensor(deriv):
    for name in ("rx", "cz"):
        with pytest.raises(ValueError):
            circuits.param_gate_tensors(name, [0.1], deriv)

"""New parameters of a compiled circuit: the rotations' tensors formed as arrays equal the
network's own conversion bit for bit, and an upload of several keys in one copy equals
one upload per key."""

import numpy as np
import pytest

from qxhip import Executor, circuits, gradients
from qxhip.circuits import Gate, gate_matrix, gate_matrix_derivative, param_gate_tensors
from qxhip.tn import TensorNetworkCircuit


@pytest.mark.parametrize("name", ["rz", "ry"])
@pytest.mark.parametrize("deriv", [False, True])
def test_rotation_tensors_equal_the_conversion(name, deriv):
    angles = [float(a) for a in np.random.default_rng(5).uniform(-10, 10, 64)] + [np.pi, 2 * np.pi, 1e-9]
    rows = param_gate_tensors(name, angles, deriv)
    for a, row in zip(angles, rows):
        g = Gate(name, (1,), a, 0)
        t = TensorNetworkCircuit(1)
        (n,) = t.push([1], gate_matrix_derivative(g) if deriv else gate_matrix(g))
        assert np.array_equal(t.tn[n].data.reshape(-1, order="F"), row)


@pytest.mark.gpu
@pytest.mark.parametrize("precision", ["c128", "c64_4m"])
def test_several_keys_in_one_copy_equal_one_at_a_time(precision):
    pc = gradients.ParamCircuit(circuits.create_param_rqc_circuit(2, 3, 3, seed=2), precision=precision, batch=4)
    one = Executor(pc.dsl, pc.graph.data, precision=precision, batch=4, graph=1)
    bits = ["010110", "110001", "001111"]
    assert np.array_equal(one.amplitudes(bits), pc.amplitudes(bits))
    keys = pc.executor.plan.keys_needed()
    pick = [len(keys) - 1, 0, len(keys) // 2]       # out of order, with others in between
    rng = np.random.default_rng(8)
    new = [rng.standard_normal(n) + 1j * rng.standard_normal(n) for k, n in pc.executor.plan.key_sizes()
           if k in {keys[i] for i in pick}]
    new = dict(zip(sorted(pick), new))
    for i in pick:
        one.update_tensor(keys[i], new[i])
    pc.executor.plan.update_tensors(np.array(pick), np.concatenate([new[i] for i in pick]))
    assert np.array_equal(one.amplitudes(bits), pc.amplitudes(bits))
    one.close()

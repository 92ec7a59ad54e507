"""A part of the slices: whole blocks of the first variables are contracted with their slices
side by side (complex128), the rest looped; either way each slice's
result enters the compensated FP64 sum."""

import ctypes as C

import numpy as np
import pytest

import qxoracle as O
import qxtest
from qxhip import Executor, _native, circuits, simulation, workloads
from test_inline_slices import data

# three variables of dims 3, 4 and 2; v1 cuts a bond of A and B, v2 one of B and C, v3 a
# bond that three tensors share
DIMS = """# version: 0.4.0
output O1 1 2
output O2 2 2
load A data_1 2,3,2
load B data_2 3,4,2
load C data_3 4,2,2
view A1 A v1 2 3
view A2 A1 v3 3 2
view B1 B v1 1 3
view B2 B1 v2 2 4
view B3 B2 v3 3 2
view C1 C v2 1 4
view C2 C1 v3 2 2
ncon D 2,3 O1 1 A2 1,2,3
ncon E 3,4 D 2,3 B3 2,4,3
ncon F 5 E 3,4 C2 4,3,5
ncon G 0 F 5 O2 5
save output G
"""

# slices of 1e16, 1, -1e16 and 0: their sum in one FP64 chain is 0, the compensated one 1
CANCEL = """# version: 0.4.0
load A data_1 4,2
load B data_2 4,2
view A1 A v1 1 4
view A2 A1 v2 2 2
view B1 B v1 1 4
view B2 B1 v2 2 2
ncon D 0 A2 1,2 B2 1,2
save output D
"""


def kept(ex):
    return next(b for b in ex.stats()["batches"] if b["active"])["kept_slices"]


def block(dims, s0, s1):
    n = 1
    for d in dims:
        if s0 % (n * d) or s1 % (n * d):
            break
        n *= d
    return n


@pytest.mark.parametrize("name", ["rqc_6x6_d12_s6", "rqc_7x7_d12_s10_open5"])
@pytest.mark.parametrize("vars_", [1, 7])
def test_saved_plans_keep_their_slices_apart(name, vars_):
    w = workloads.WORKLOADS[name]
    dsl = w.load()[0]
    plain = _native.inspect(dsl, batch=8, batch_last=bool(w.batch_last))
    info = _native.inspect(dsl, batch=8, fused=vars_, kept=True, batch_last=bool(w.batch_last))
    assert info["kept_slices"] == vars_ + 1 and info["result_elems"] == plain["result_elems"]


@pytest.mark.gpu
@pytest.mark.parametrize("options", [{}, {"graph": 1}, {"autotune": 1, "graph": 1}, {"profile": 1}, {"batch_last": 1}])
def test_every_range_of_variables_of_other_dims(options):
    values = data(DIMS)
    ex = Executor(DIMS, values, batch=16, **options)
    every = list(O.slice_assignments(O.parse(DIMS)))
    assert ex.num_slices == 24
    for s0 in range(24):
        for s1 in range(s0 + 1, 25):
            ref = O.amplitudes(DIMS, values, ["01", "+1", "10"], slices=every[s0:s1])
            for _ in range(2):
                got = np.asarray(ex.amplitudes(["01", "+1", "10"], s0, s1)).reshape(-1)
                assert np.max(np.abs(got - ref.reshape(-1))) <= 1e-12 * np.max(np.abs(ref)), (s0, s1)
            assert kept(ex) == (1 if (s0, s1) == (0, 24) else block((3, 4, 2), s0, s1)), (s0, s1)
    ex.close()


@pytest.mark.gpu
@pytest.mark.parametrize("precision", ["c128", "c64_4m"])
def test_ranges_of_a_sliced_circuit(precision):
    circ = circuits.create_rqc_circuit(2, 3, 6, seed=21)
    _, _, g = qxtest.graph_for(circ, planner="greedy", nslice=3)
    dsl, values, bits = g.to_dsl(), g.data, simulation.amplitudes_uniform(6, 99, 5)
    ex = Executor(dsl, values, precision=precision, batch=64, graph=1)
    looped = Executor(dsl, values, precision=precision, batch=64, graph=1, fuse_slices=0)
    for s0 in range(8):
        for s1 in range(s0 + 1, 9):
            a, b = ex.amplitudes(bits, s0, s1), looped.amplitudes(bits, s0, s1)
            if precision == "c128":
                assert np.max(np.abs(a - b)) <= 1e-12 * np.max(np.abs(b)), (s0, s1)
            elif (s0, s1) != (0, 8):
                assert np.array_equal(a, b), (s0, s1)
    ex.close()
    looped.close()


@pytest.mark.gpu
@pytest.mark.parametrize("batch", [1, 4])
def test_the_sum_of_a_part_is_compensated(batch):
    values = {"data_1": np.zeros((4, 2), dtype=np.complex128), "data_2": np.ones((4, 2), dtype=np.complex128)}
    values["data_1"][:, 0] = [1e16, 1.0, -1e16, 0.0]
    values["data_1"][:, 1] = [1e16j, -1e16j, 2j, 0.0]
    ex = Executor(CANCEL, values, batch=batch)
    assert ex.amplitudes([""], 0, 4).reshape(-1)[0] == 1.0
    assert kept(ex) == 4
    assert ex.amplitudes([""], 4, 8).reshape(-1)[0] == 2.0j
    ex.close()


@pytest.mark.gpu
def test_allocation_free_parts_do_not_depend_on_earlier_calls():
    """The allocation-free call of a range returns the same bits whatever ranges were called
    before it."""
    circ = circuits.create_rqc_circuit(2, 3, 6, seed=21)
    _, _, g = qxtest.graph_for(circ, planner="greedy", nslice=3)
    bits = simulation.amplitudes_uniform(6, 99, 4)
    f = _native.lib().qx_amplitudes_noalloc
    got = {}
    for before in ([(0, 8), (3, 5)], [(4, 8)], [(2, 4), (4, 8), (0, 2)]):
        ex = Executor(g.to_dsl(), g.data, batch=4)
        for r in before:
            ex.amplitudes(bits, *r)
        for s0, s1 in ((4, 8), (2, 4), (3, 6)):
            out = np.zeros(4, dtype=np.complex128)
            assert f(ex.plan._h, ex.plan._bits(bits), 4, s0, s1, out.ctypes.data_as(C.POINTER(C.c_double))) == 0
            assert np.array_equal(out, got.setdefault((s0, s1), out)), (before, s0, s1)
            want = ex.amplitudes(bits, s0, s1)
            assert np.max(np.abs(out - want)) <= 1e-12 * np.max(np.abs(want)), (before, s0, s1)
        ex.close()

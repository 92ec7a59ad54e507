"""Every range of slices of a plan, those that are whole blocks of the first variables
(contracted inline) and the others (looped), against the same plan with every slice
looped and against the oracle's slices; also without allocations after either kind."""

import ctypes as C

import numpy as np
import pytest

import qxoracle as O
import qxtest
from qxhip import Executor, _native, circuits, simulation

pytestmark = pytest.mark.gpu


def _plan():
    circ = circuits.create_rqc_circuit(2, 3, 6, seed=21)
    _, _, g = qxtest.graph_for(circ, planner="greedy", nslice=3)
    return g.to_dsl(), g.data, simulation.amplitudes_uniform(6, 99, 5)


@pytest.mark.parametrize("precision,graph", [("c128", 0), ("c128", 1), ("c64_4m", 1)])
def test_every_range_equals_the_looped_one(precision, graph):
    dsl, data, bits = _plan()
    ex = Executor(dsl, data, precision=precision, batch=4, graph=graph)
    looped = Executor(dsl, data, precision=precision, batch=4, graph=graph, fuse_slices=0)
    assert ex.num_slices == 8
    every = list(O.slice_assignments(O.parse(dsl)))
    eps = 1e-12 if precision == "c128" else 1e-4
    for s0 in range(8):
        for s1 in range(s0 + 1, 9):
            a, b = ex.amplitudes(bits, s0, s1), looped.amplitudes(bits, s0, s1)
            ref = O.amplitudes(dsl, data, bits, slices=every[s0:s1])
            scale = np.max(np.abs(ref))
            assert np.max(np.abs(a - b)) <= eps * scale, (s0, s1)
            assert np.max(np.abs(a - ref)) <= eps * scale, (s0, s1)
            if precision != "c128" and (s0, s1) != (0, 8):   # complex64 keeps the FP64 sum of slices
                assert np.array_equal(a, b), (s0, s1)
    ex.close()
    looped.close()


def test_ranges_without_allocations_after_an_inline_one():
    dsl, data, bits = _plan()
    ex = Executor(dsl, data, batch=4)
    whole = ex.amplitudes(bits[:4], 4, 8)            # whole blocks: inline
    f = _native.lib().qx_amplitudes_noalloc
    for s0, s1, ref in ((4, 8, whole), (4, 8, whole), (3, 6, None), (2, 4, None)):
        out = np.zeros(4, dtype=np.complex128)
        assert f(ex.plan._h, ex.plan._bits(bits[:4]), 4, s0, s1, out.ctypes.data_as(C.POINTER(C.c_double))) == 0
        r = O.amplitudes(dsl, data, bits[:4], slices=list(O.slice_assignments(O.parse(dsl)))[s0:s1])
        assert np.max(np.abs(out - r)) <= 1e-12 * np.max(np.abs(r))
        assert ref is None or np.array_equal(out, ref)
    ex.close()

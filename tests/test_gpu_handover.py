"""Calls whose bitstrings and results go through pinned host memory, and those just too
large for it: equal values on both sides of each limit, eagerly and replayed."""

import numpy as np
import pytest

import qxoracle as O
from qxhip import Executor, simulation, workloads

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("graph", [0, 1])
def test_bitstrings_up_to_and_beyond_the_pinned_area(graph):
    dsl, data, _ = workloads.WORKLOADS["rqc_3x3_d16"].load()
    ex = Executor(dsl, data, graph=graph)
    table = dict(zip(simulation.amplitudes_all(9), O.amplitudes(dsl, data, list(simulation.amplitudes_all(9)))))
    for seed, n in ((1, 455), (2, 456), (3, 455), (4, 1)):     # 4095 and 4104 bytes of bitstrings
        draws = np.random.default_rng(seed).integers(0, 2, size=(n, 9))
        bits = ["".join("01"[b] for b in row) for row in draws]
        ref = np.array([table[b] for b in bits])
        assert np.max(np.abs(ex.amplitudes(bits) - ref) / np.abs(ref)) <= 1e-12
    ex.close()


def test_samples_beyond_the_pinned_area_start_with_the_same_ones():
    dsl, data, _ = workloads.WORKLOADS["rqc_3x3_d16"].load()
    ex = Executor(dsl, data, graph=1)
    few_bits, few_amps, _, _ = ex.sample_rejection(300, 5)
    bits, amps, _, used = ex.sample_rejection(10400, 5)        # 25 bytes each: over 257792
    assert len(bits) == 10400 and used >= 10400
    assert bits[:300] == few_bits and np.array_equal(amps[:300], few_amps)
    ex.close()

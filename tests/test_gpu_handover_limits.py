"""Results and gradients on both sides of the limits of the pinned block that small calls hand
over through: 16112 results of a forward call, 8056 amplitudes and 8056 gradient values of a
pullback; eager and replayed."""

import numpy as np
import pytest

import qxoracle as O
from qxhip import Executor, simulation, workloads

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def plan_3x3():
    dsl, data, _ = workloads.WORKLOADS["rqc_3x3_d16"].load()
    every = list(simulation.amplitudes_all(9))
    return dsl, data, dict(zip(every, O.amplitudes(dsl, data, every)))


def bitstrings(n, seed):
    return ["".join("01"[b] for b in row) for row in np.random.default_rng(seed).integers(0, 2, size=(n, 9))]


@pytest.mark.parametrize("graph", [0, 1])
def test_results_up_to_and_beyond_the_pinned_area(plan_3x3, graph):
    dsl, data, table = plan_3x3
    ex = Executor(dsl, data, graph=graph)
    for seed, n in ((1, 16112), (2, 16113), (3, 16112), (4, 16113), (5, 3)):
        bits = bitstrings(n, seed)
        ref = np.array([table[b] for b in bits])
        assert np.max(np.abs(ex.amplitudes(bits) - ref) / np.abs(ref)) <= 1e-12
    ex.close()


@pytest.mark.parametrize("graph", [0, 1])
def test_pullback_amplitudes_up_to_and_beyond_their_half(plan_3x3, graph):
    dsl, data, table = plan_3x3
    ex = Executor(dsl, data, graph=graph)
    for seed, n in ((1, 8056), (2, 8057), (3, 8056), (4, 2)):
        bits = bitstrings(n, seed)
        ref = np.array([table[b] for b in bits])
        amps, grad = ex.plan.norm_vjp(bits)
        assert np.max(np.abs(amps.reshape(-1) - ref) / np.abs(ref)) <= 1e-12
        # the pullback is linear in its cotangent, which is 2 amp here
        again = ex.plan.vjp(bits, 2 * ref)
        for k in again:
            want = np.asarray(again[k]).reshape(-1)
            got = np.asarray(grad[k]).reshape(-1)
            assert np.max(np.abs(got - want)) <= 1e-10 * np.max(np.abs(want)), k
    ex.close()


@pytest.mark.parametrize("graph", [0, 1])
@pytest.mark.parametrize("extra", [1, 2])
def test_gradients_up_to_and_beyond_their_half(graph, extra):
    """amp[b, s] = sum over i, k of v_b[i] A[i, k] B[k] S[s]; 3 x 2685 + extra gradient values."""
    n = 2685
    dsl = f"""# version: 0.4.0
output O1 1 2
load A data_a 2,{n}
load B data_b {n}
load S data_s {extra}
ncon D 2 O1 1 A 1,2
ncon E 0 D 2 B 2
ncon F 3 E 0 S 3
save output F
"""
    rng = np.random.default_rng(extra)
    cplx = lambda *s: rng.normal(size=s) + 1j * rng.normal(size=s)   # noqa: E731
    a, b, s = cplx(2, n), cplx(n), cplx(extra)
    ex = Executor(dsl, {"data_a": a, "data_b": b, "data_s": s}, batch=4, graph=graph)
    v = np.array([[1, 0], [0, 1], [np.sqrt(0.5), -np.sqrt(0.5)]])
    for _ in range(3):
        cot = cplx(3, extra)
        g = ex.vjp(["0", "1", "-"], cot)
        c = v.T @ (cot @ s.conj())                                    # over i
        want = {"data_a": np.outer(c, b.conj()), "data_b": a.conj().T @ c,
                "data_s": cot.T @ (v @ (a @ b)).conj()}
        for k, w in want.items():
            got = np.asarray(g[k]).reshape(w.shape, order="F")
            assert np.max(np.abs(got - w)) <= 1e-11 * np.max(np.abs(w)), k
    ex.close()

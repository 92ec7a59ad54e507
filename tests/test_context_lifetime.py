"""A context that is destroyed before its plans: the plans' later calls and their own
destruction must not reach freed memory."""

import numpy as np
import pytest

import qxoracle as O
from qxhip import _native, simulation, workloads
from test_sanitize import _run, san_env  # noqa: F401


@pytest.mark.parametrize("args", [("rqc_3x3_d16", "--graph", "1", "--vjp", "--noalloc"), ("sliced", "--calls", "0")])
def test_plan_outlives_its_context_under_sanitizers(san_env, args):  # noqa: F811
    _run(san_env, *args, "--close-context-first")


@pytest.mark.gpu
def test_plan_outlives_its_context():
    dsl, data, _ = workloads.WORKLOADS["rqc_3x3_d16"].load()
    bits = simulation.amplitudes_uniform(9, 3, 8)
    ref = O.amplitudes(dsl, data, bits)
    ctx = _native.Context()          # (not the process's shared one)
    plan = _native.Plan(ctx, dsl, data, graph=1)
    plan.amplitudes(bits)
    ctx.close()
    for _ in range(3):
        assert np.max(np.abs(plan.amplitudes(bits) - ref) / np.abs(ref)) <= 1e-12
    plan.close()

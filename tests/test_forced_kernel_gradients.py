"""Pullbacks with every kernel forced in turn (plan option `kernel`), on steps with a narrow
operand, whose backward steps the row kernel runs over the other side."""

import os
import subprocess
import sys

import numpy as np
import pytest

from qxhip import Executor
from test_sanitize import ROOT, san_env  # noqa: F401
from test_tuning_operands import narrow

SHAPES = [(2, 12, 1), (4, 12, 3), (6, 9, 4), (1, 10, 2)]


def test_backward_steps_read_inside_the_operands(san_env):  # noqa: F811
    code = """
import sys
sys.path[:0] = [%r, %r, %r]
import numpy as np
from test_forced_kernel_gradients import SHAPES, narrow
from qxhip import Executor
for shape in SHAPES:
    dsl, data = narrow(*shape)
    for kernel in range(13):
        ex = Executor(dsl, data, batch=1, kernel=kernel)
        ex.vjp([""], np.ones((1, ex.plan.result_elems), dtype=np.complex128))
        ex.close()
print("sequence done")
""" % tuple(os.path.join(ROOT, d) for d in ("tests", "oracle", "qxtools.jl_amd"))
    r = subprocess.run([sys.executable, "-c", code], env=san_env, capture_output=True, text=True, timeout=300)
    assert r.returncode == 0 and "sequence done" in r.stdout, r.stderr[-3000:]


@pytest.mark.gpu
@pytest.mark.parametrize("kernel", range(13))
@pytest.mark.parametrize("nm,nn,nk", SHAPES)
def test_gradients_with_a_forced_kernel(nm, nn, nk, kernel):
    dsl, data = narrow(nm, nn, nk)
    rng = np.random.default_rng(kernel)
    ex = Executor(dsl, data, batch=1, kernel=kernel)
    cot = rng.normal(size=(1, ex.plan.result_elems)) + 1j * rng.normal(size=(1, ex.plan.result_elems))
    g = ex.vjp([""], cot)
    ex.close()
    # C's legs: the first of M, all of N, the rest of M
    c = cot.reshape([2] * (nm + nn), order="F")
    c = np.moveaxis(c, range(1, nn + 1), range(nm, nm + nn)).reshape(2 ** nm, 2 ** nn, order="F")
    a = data["data_2"].reshape(2 ** nm, 2 ** nk, order="F")
    b = data["data_1"].reshape(2 ** nk, 2 ** nn, order="F")
    for key, want in (("data_2", c @ b.conj().T), ("data_1", a.conj().T @ c)):
        got = np.asarray(g[key]).reshape(want.shape, order="F")
        assert np.max(np.abs(got - want)) <= 1e-12 * np.max(np.abs(want)), key

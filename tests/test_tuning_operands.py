"""The autotuner's candidates that exchange a step's operands: the tuning call reads each
operand where it lies and returns the amplitudes."""

import os
import subprocess
import sys

import numpy as np
import pytest

import qxoracle as O
from qxhip import Executor, _native
from test_sanitize import ROOT, san_env  # noqa: F401

# (M, N, K) bits: a narrow A against a long B, A the last of the data
SHAPES = [(2, 12, 1), (2, 13, 2), (4, 12, 3), (6, 12, 4), (1, 14, 1)]


def narrow(nm, nn, nk):
    legs = list(range(1, nm + nn + nk + 1))
    m, n, k = legs[:nm], legs[nm:nm + nn], legs[nm + nn:]
    fmt = lambda ls: ",".join(map(str, ls))   # noqa: E731
    dsl = "\n".join(["# version: 0.4.0", f"load B data_1 {fmt([2] * (nk + nn))}", f"load A data_2 {fmt([2] * (nm + nk))}",
                     f"ncon C {fmt(m[:1] + n + m[1:])} A {fmt(m + k)} B {fmt(k + n)}", "save output C"]) + "\n"
    rng = np.random.default_rng(nn)
    cplx = lambda r: rng.normal(size=[2] * r) + 1j * rng.normal(size=[2] * r)   # noqa: E731
    return dsl, {"data_1": cplx(nk + nn), "data_2": cplx(nm + nk)}


@pytest.mark.parametrize("nm,nn,nk", SHAPES)
def test_candidates_exchange_the_operands(nm, nn, nk):
    (step,) = _native.inspect(narrow(nm, nn, nk)[0])["steps"]
    assert any("swap" in c for c in step["candidates"])


def test_tuning_reads_inside_the_operands(san_env):  # noqa: F811
    code = """
import sys
sys.path[:0] = [%r, %r, %r]
from test_tuning_operands import SHAPES, narrow
from qxhip import Executor
for shape in SHAPES:
    dsl, data = narrow(*shape)
    for precision in ("c128", "c64_4m"):
        ex = Executor(dsl, data, precision=precision, batch=1, autotune=1, graph=1)
        for _ in range(3):
            ex.amplitudes([""])
        ex.close()
print("sequence done")
""" % tuple(os.path.join(ROOT, d) for d in ("tests", "oracle", "qxtools.jl_amd"))
    r = subprocess.run([sys.executable, "-c", code], env=san_env, capture_output=True, text=True, timeout=300)
    assert r.returncode == 0 and "sequence done" in r.stdout, r.stderr[-3000:]


@pytest.mark.gpu
@pytest.mark.parametrize("precision,tol", [("c128", 1e-13), ("c64_4m", 1e-5)])
@pytest.mark.parametrize("nm,nn,nk", SHAPES)
def test_the_tuning_call_returns_the_amplitudes(nm, nn, nk, precision, tol):
    dsl, data = narrow(nm, nn, nk)
    ref = O.amplitudes(dsl, data, [""])[0].reshape(-1, order="F")
    ex = Executor(dsl, data, precision=precision, batch=1, autotune=1, graph=1)
    for call in range(3):
        got = np.asarray(ex.amplitudes([""])).reshape(-1)
        assert np.max(np.abs(got - ref)) <= tol * np.max(np.abs(ref)), call
    ex.close()

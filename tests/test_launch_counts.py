"""`last_call_launches` of qx_plan_stats, which also decides what is captured, against the
launches that the simulated device of the sanitizer build counts."""

import os
import subprocess
import sys

import pytest

from test_sanitize import ROOT, san_env  # noqa: F401

CODE = """
import ctypes, sys
sys.path[:0] = [%r, %r, %r]
import numpy as np
import qxtest
from qxhip import Executor, _native, circuits, simulation, workloads
lib = _native.lib()
lib.qx_sim_launches.restype = ctypes.c_int64

def count(what, ex, call):
    call()
    before = lib.qx_sim_launches()
    call()
    ran, said = lib.qx_sim_launches() - before, ex.stats()["last_call_launches"]
    print(what, ran, said, flush=True)
    assert ran == said, what

name, options = sys.argv[1], eval(sys.argv[2])
if name == "slices":
    circ = circuits.create_rqc_circuit(3, 3, 10, seed=21)
    _, _, g = qxtest.graph_for(circ, planner="greedy", nslice=8)
    dsl, data, bits = g.to_dsl(), g.data, simulation.amplitudes_uniform(9, 7, 32)
else:
    dsl, data, bits = workloads.WORKLOADS[name].load()
    bits = bits[:8]
ex = Executor(dsl, data, **options)
count("all", ex, lambda: ex.amplitudes(bits))
if ex.num_slices > 8:
    count("block", ex, lambda: ex.amplitudes(bits, 4, 8))
    count("odd", ex, lambda: ex.amplitudes(bits, 3, 6))
if "vjp" in sys.argv[3:]:
    cot = np.ones(len(bits), dtype=np.complex128)
    count("vjp", ex, lambda: ex.vjp(bits, cot))
print("cap", ex.stats()["max_graph_launches"])
""" % tuple(os.path.join(ROOT, d) for d in ("tests", "oracle", "qxtools.jl_amd"))


@pytest.mark.parametrize("name,options,more", [
    ("slices", "dict(batch=4, graph=1, fuse_slices=0)", "vjp"),
    ("slices", "dict(batch=64, graph=1)", "vjp"),
    ("slices", "dict(batch=4, small_walk=1)", ""),
    ("slices", "dict(batch=4, kernel=6, chains=0)", ""),
    ("rqc_3x3_d16", "dict(graph=1)", "vjp"),
    ("rqc_5x5_d20", "dict(autotune=1, graph=1)", ""),
    ("rqc_6x6_d12_s6", "dict(precision='c64_4m')", ""),
    ("rqc_6x6_d12_s6", "dict(kernel=5, graph=1)", ""),
    ("rqc_7x7_d12_s10_open5", "dict(precision='c64_bf16x3', kernel=10)", ""),
])
def test_reported_launches(san_env, name, options, more):  # noqa: F811
    r = subprocess.run([sys.executable, "-c", CODE, name, options, more], env=san_env, capture_output=True, text=True,
                       timeout=600)
    assert r.returncode == 0, r.stdout + r.stderr[-3000:]
    # the looped call that tests/test_gpu_graph.py runs as one beyond the capture limit
    if "fuse_slices=0" in options:
        ran, cap = int(r.stdout.split("all ")[1].split()[0]), int(r.stdout.split("cap ")[1])
        assert ran > cap

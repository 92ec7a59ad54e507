"""Slice variables whose sum is not one contraction with their legs left whole: a variable
that cuts two bonds, one that fixes a leg of the saved tensor, one that no contraction
sums.  Every range of their slices against the oracle's loop."""

import os
import subprocess
import sys

import numpy as np
import pytest

import qxoracle as O
from qxhip import Executor, _native, workloads
from test_sanitize import ROOT, san_env  # noqa: F401

HEAD = """# version: 0.4.0
output O1 1 2
load A data_1 2,2,4
load B data_2 2,4,2
load C data_3 2,2
"""
# bonds x (A-B, dim 4) and y (B-C, dim 2), A's leg 1 the output; variables v1, v2
PROGRAMS = {
    "one_bond": (HEAD + """view A1 A v1 3 4
view B1 B v1 2 4
ncon D 2,3 O1 1 A1 1,2,3
ncon E 2,5,6 D 2,3 B1 5,3,6
ncon F 2,5 E 2,5,6 C 6,7
save output F
""").replace("C 6,7", "V 6").replace("load C data_3 2,2", "load V data_4 2"),
    "two_bonds": HEAD.replace("load A data_1 2,2,4", "load A data_1 2,2,2").replace("load B data_2 2,4,2", "load B data_2 2,2,2") +
    """view A1 A v1 3 2
view B1 B v1 2 2
view B2 B1 v1 3 2
view C1 C v1 1 2
ncon D 2,3 O1 1 A1 1,2,3
ncon E 2,5,6 D 2,3 B2 5,3,6
ncon F 2,5,7 E 2,5,6 C1 6,7
save output F
""",
    "two_apart": HEAD.replace("load A data_1 2,2,4", "load A data_1 2,2,2").replace("load B data_2 2,4,2", "load B data_2 2,2,2") +
    """view A1 A v1 3 2
view B1 B v1 2 2
load G data_5 2,2
load H data_6 2,2
view G1 G v1 2 2
view H1 H v1 1 2
ncon D 2,3 O1 1 A1 1,2,3
ncon E 2,5,6 D 2,3 B1 5,3,6
ncon I 8,9 G1 8,4 H1 4,9
ncon F 2,5,7 E 2,5,6 C 6,7
ncon J 2,5,7,8,9 F 2,5,7 I 8,9
save output J
""",
    "saved_leg": HEAD + """view A1 A v1 2 2
view A2 A1 v2 3 4
view B1 B v2 2 4
ncon D 2,3 O1 1 A2 1,2,3
ncon E 2,5,6 D 2,3 B1 5,3,6
ncon F 2,5,7 E 2,5,6 C 6,7
save output F
""",
    "unsummed": HEAD + """load G data_5 2,2
view G1 G v1 1 2
ncon D 2,3 O1 1 A 1,2,3
ncon E 2,5,6 D 2,3 B 5,3,6
ncon F 2,5,7 E 2,5,6 C 6,7
save output F
""",
    "unused_sum": HEAD + """load G data_5 2,2
load H data_6 2
view G1 G v1 1 2
view H1 H v1 1 2
ncon I 2 G1 1,2 H1 1
ncon D 2,3 O1 1 A 1,2,3
ncon E 2,5,6 D 2,3 B 5,3,6
ncon F 2,5,7 E 2,5,6 C 6,7
save output F
""",
}
INLINE = {"one_bond": 1, "two_bonds": 0, "two_apart": 0, "saved_leg": 2, "unsummed": 0, "unused_sum": 0}


def data(dsl, seed=3):
    rng = np.random.default_rng(seed)
    out = {}
    for f in (s.split() for s in dsl.splitlines() if s.startswith("load")):
        shape = [int(x) for x in f[3].split(",")]
        out[f[2]] = rng.normal(size=shape) + 1j * rng.normal(size=shape)
    return out


@pytest.mark.parametrize("name", PROGRAMS)
def test_variables_that_may_be_summed_inline(name):
    assert _native.inspect(PROGRAMS[name])["inline_vars"] == INLINE[name]


@pytest.mark.parametrize("name", ["rqc_6x6_d12_s6", "rqc_7x7_d12_s10_open5"])
def test_saved_plans_sum_every_variable_inline(name):
    dsl = workloads.WORKLOADS[name].load()[0]
    n = len({s.split()[3] for s in dsl.splitlines() if s.startswith("view")})
    assert _native.inspect(dsl)["inline_vars"] == (1 << n) - 1


def test_results_stay_inside_the_callers_buffer(san_env):  # noqa: F811
    """A saved tensor's sliced leg has one value per call; the sanitizer sees a write of more."""
    code = """
import sys
sys.path[:0] = [%r, %r, %r]
from test_inline_slices import PROGRAMS, data
from qxhip import Executor
ex = Executor(PROGRAMS["saved_leg"], data(PROGRAMS["saved_leg"]), batch=4)
for s0, s1 in ((0, 8), (0, 2), (2, 8), (1, 3)):
    ex.amplitudes(["0"], s0, s1)
ex.close()
print("sequence done")
""" % tuple(os.path.join(ROOT, d) for d in ("tests", "oracle", "qxtools.jl_amd"))
    r = subprocess.run([sys.executable, "-c", code], env=san_env, capture_output=True, text=True, timeout=300)
    assert r.returncode == 0 and "sequence done" in r.stdout, r.stderr[-3000:]


@pytest.mark.gpu
@pytest.mark.parametrize("batch", [1, 8])
@pytest.mark.parametrize("name", PROGRAMS)
def test_every_range_equals_the_oracles_loop(name, batch):
    dsl = PROGRAMS[name]
    values = data(dsl)
    ex = Executor(dsl, values, batch=batch)
    every = list(O.slice_assignments(O.parse(dsl)))
    assert ex.num_slices == len(every)
    for s0 in range(len(every)):
        for s1 in range(s0 + 1, len(every) + 1):
            for bits in (["1"], ["0", "+", "-"]):
                got = np.asarray(ex.amplitudes(bits, s0, s1))
                ref = O.amplitudes(dsl, values, bits, slices=every[s0:s1])
                assert got.size == ref.size
                ref = np.stack([r.reshape(-1, order="F") for r in ref])
                assert np.max(np.abs(got.reshape(len(bits), -1) - ref)) <= 1e-12 * np.max(np.abs(ref)), (s0, s1)
    ex.close()

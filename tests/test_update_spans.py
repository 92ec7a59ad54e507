"""New values of some data keys: what is copied to the device is about those keys' bytes,
whatever lies between them."""

import os
import subprocess
import sys

import numpy as np
import pytest

import qxoracle as O
from qxhip import Executor
from test_sanitize import ROOT, san_env  # noqa: F401

# small keys around one of 2^16 values (1 MiB)
DSL = """# version: 0.4.0
load A data_a 2
load B data_b 2,256,128
load C data_c 256
load D data_d 128
load E data_e 2
ncon F 2,3 A 1 B 1,2,3
ncon G 3 F 2,3 C 2
ncon H 0 G 3 D 3
ncon I 1 H 0 E 1
save output I
"""
SIZES = {"data_a": (2,), "data_b": (2, 256, 128), "data_c": (256,), "data_d": (128,), "data_e": (2,)}


def values(seed):
    rng = np.random.default_rng(seed)
    return {k: rng.normal(size=s) + 1j * rng.normal(size=s) for k, s in SIZES.items()}


@pytest.mark.parametrize("picked,most", [((0, 4), 32 + 32 + 8192), ((4, 0, 2), 3 * 4096 + 8192), ((2, 3), 12288),
                                         ((0, 1), 2 * 2 ** 20 + 4096), ((3,), 4096)])
def test_bytes_copied(san_env, picked, most):  # noqa: F811
    code = """
import ctypes, sys
sys.path[:0] = [%r, %r, %r]
import numpy as np
from test_update_spans import DSL, SIZES, values
from qxhip import Executor, _native
up = _native.lib().qx_sim_uploaded
up.restype = ctypes.c_int64
ex = Executor(DSL, values(1), batch=1)
names = ex.plan.keys_needed()
before = up()
ex.plan.update_tensors(np.array(%r), np.concatenate([values(2)[names[i]].reshape(-1, order="F") for i in %r]))
print("copied", up() - before)
""" % (*(os.path.join(ROOT, d) for d in ("tests", "oracle", "qxtools.jl_amd")), picked, picked)
    r = subprocess.run([sys.executable, "-c", code], env=san_env, capture_output=True, text=True, timeout=300)
    assert r.returncode == 0, r.stderr[-3000:]
    assert int(r.stdout.split("copied")[1]) <= most


@pytest.mark.gpu
@pytest.mark.parametrize("precision,tol", [("c128", 1e-12), ("c64_4m", 1e-4)])
def test_every_pick_reaches_the_device(precision, tol):
    ex = Executor(DSL, values(1), precision=precision, batch=1)
    now, names = values(1), ex.plan.keys_needed()
    for step, picked in enumerate([(0, 4), (4, 0, 2), (2, 3), (1,), (3, 1, 0), (0, 1, 2, 3, 4)]):
        new = values(10 + step)
        ex.plan.update_tensors(np.array(picked), np.concatenate([new[names[i]].reshape(-1, order="F") for i in picked]))
        now.update({names[i]: new[names[i]] for i in picked})
        ref = O.amplitudes(DSL, now, [""]).reshape(-1)
        got = np.asarray(ex.amplitudes([""])).reshape(-1)
        assert np.max(np.abs(got - ref)) <= tol * np.max(np.abs(ref)), picked
    ex.close()

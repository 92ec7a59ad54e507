"""QX_C64_3M takes three real products per complex product only on GEMM steps whose FP32
products bind (both sides >= 64, K >= 32); every other step computes what QX_C64_4M does."""

import numpy as np
import pytest

from qxhip import Executor, _native
from test_gemm_grid import gemm_steps
from test_gpu_kernels import plain_step

SHAPES = [((10, 5, 8, 3), 4), ((12, 3, 9, 2), 4), ((4, 6, 6, 4), 4), ((4, 6, 6, 5), 3), ((4, 5, 7, 6), 4),
          ((0, 7, 6, 7), 3)]


@pytest.mark.parametrize("shape,products", SHAPES)
def test_products_by_shape(shape, products):
    dsl, _, _ = plain_step(1, *shape, 0, 0, 0)
    (g,) = gemm_steps(_native.inspect(dsl, "c64_3m")["steps"])
    assert g["products"] == products
    (g,) = gemm_steps(_native.inspect(dsl, "c64_4m")["steps"])
    assert g["products"] == 4


@pytest.mark.parametrize("name", ["rqc_5x5_d20", "rqc_6x6_d12_s6"])
def test_saved_plans_take_three_only_on_large_steps(name):
    from qxhip import workloads

    dsl = workloads.WORKLOADS[name].load()[0]
    steps = gemm_steps(_native.inspect(dsl, "c64_3m", batch=256, fused=63)["steps"])
    for s in steps:
        assert (s["products"] == 3) == (s["M"] >= 64 and s["N"] >= 64 and s["K"] >= 32), s["name"]


@pytest.mark.gpu
@pytest.mark.parametrize("shape,products", [x for x in SHAPES if x[1] == 4])
def test_other_steps_equal_four_products(shape, products):
    dsl, data, _ = plain_step(2, *shape, 1, 0, 0)
    got = []
    for precision in ("c64_3m", "c64_4m"):
        ex = Executor(dsl, data, precision=precision, batch=1, kernel=5)
        got.append(np.asarray(ex.amplitudes([""])).reshape(-1))
        ex.close()
    assert np.array_equal(*got)

"""The any-layout matrix-core GEMM's tiles of 128 rows or columns against a complex128
product, in each operand order."""

import numpy as np
import pytest

from qxhip import Executor
from test_gpu_kernels import plain_step

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape,layout", [((10, 7, 6, 6), 0), ((10, 6, 7, 6), 3), ((9, 7, 7, 6), 5)])
def test_wide_tiles(shape, layout):
    dsl, data, ref = plain_step(41 + layout, *shape, layout & 1, layout >> 1 & 1, layout >> 2)
    ex = Executor(dsl, data, precision="c64_4m", batch=1, kernel=5)
    got = np.asarray(ex.amplitudes([""])).reshape(-1)
    ex.close()
    assert np.linalg.norm(got - ref) <= 5e-6 * np.linalg.norm(ref)

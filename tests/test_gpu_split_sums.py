"""Sums of K-split partials with several lanes per element: long contractions into few
values, with counts of values and partials on both sides of a workgroup's 16 by 16."""

import numpy as np
import pytest

from qxhip import Executor
from test_gpu_kernels import plain_step

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision,tol", [("c128", 1e-12), ("c64_4m", 1e-4)])
@pytest.mark.parametrize("nm,nn,nk", [(1, 0, 17), (0, 2, 16), (2, 2, 15), (3, 2, 16), (5, 4, 14), (4, 4, 18)])
@pytest.mark.parametrize("kernel", [-1, 0, 5, 6])
def test_long_contractions_into_few_values(nm, nn, nk, precision, tol, kernel):
    dsl, data, ref = plain_step(61, 0, nm, nn, nk, 0, 0, 0)
    ex = Executor(dsl, data, precision=precision, batch=1, kernel=kernel)
    got = np.asarray(ex.amplitudes([""])).reshape(-1)
    assert np.max(np.abs(got - ref)) <= tol * np.max(np.abs(ref))
    ex.close()

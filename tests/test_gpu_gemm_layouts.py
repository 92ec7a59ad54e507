"""The matrix-core GEMM on operands of any layout (k_contract_gemm_mfma): every tile
shape, tiles with fewer rows, columns or k values than their shape, K splits, hyper legs
between the others, both orientations of the result, against the oracle's TTGT product.
Tolerances as for the other kernels: 1e-12 complex128, 2e-5 complex64 (FP32 sums)."""

import numpy as np
import pytest

from test_gpu_kernels import err, single_step

pytestmark = pytest.mark.gpu

# legs of H, M, N, K: 64 x 64 tiles, the narrower shapes either way round, fewer values
# than a tile or a stage has, one value, a long K split over workgroups, many units
SHAPES = [(0, 6, 6, 4), (2, 7, 8, 5), (1, 5, 9, 4), (1, 9, 5, 3), (3, 4, 9, 6), (2, 9, 4, 2), (1, 2, 8, 1),
          (1, 8, 1, 5), (0, 3, 3, 0), (0, 1, 1, 12), (4, 6, 6, 7), (0, 4, 4, 11), (6, 7, 6, 3), (2, 6, 7, 0),
          (3, 0, 7, 4), (5, 6, 9, 2)]


@pytest.mark.parametrize("shape", SHAPES)
@pytest.mark.parametrize("kernel", [5, 7])
@pytest.mark.parametrize("prec,tol", [("c128", 1e-12), ("c64_4m", 2e-5), ("c64_3m", 5e-5)])
def test_any_layout(shape, kernel, prec, tol):
    from qxhip import Executor

    for seed in (0, 1, 2):   # three random leg orders
        dsl, data, ref = single_step(7000 + 31 * seed + sum(3 ** i * n for i, n in enumerate(shape)), *shape)
        ex = Executor(dsl, data, precision=prec, kernel=kernel)
        out = np.asarray(ex.amplitudes([""])).reshape(-1)
        st = next(b for b in ex.stats()["batches"] if b["active"])["steps"][0]
        ex.close()
        assert st["variant"] == ("k_contract_gemm_mfma" if kernel == 5 else "k_contract_gemm_mfma<yx>")
        assert err(out, ref) < tol, (seed, err(out, ref))

"""The matrix-core GEMM's launch grid: fewer than 2^32 lanes whatever the step's batch
dimension, the units beyond that walked by the workgroups."""

import numpy as np
import pytest

from qxhip import Executor, _native
from test_gpu_kernels import plain_step


def batched_gemm(nh, nm, nn, nk, seed=0):
    """C[n m h] = A[m k h] B[k n h], N fastest in C, both operands outer products of small
    factors (formed on the device) and C summed over h against a third, so that a step with
    2^28 results needs a few hundred input values; the sum by the factors."""
    rng = np.random.default_rng(seed)
    legs = iter(range(1, 200))
    H, M, N, K = ([next(legs) for _ in range(n)] for n in (nh, nm, nn, nk))
    fmt = lambda ls: ",".join(map(str, ls))   # noqa: E731
    lines, data = ["# version: 0.4.0"], {}

    def load(name, n):
        data["data_" + name] = rng.normal(size=[2] * n) + 1j * rng.normal(size=[2] * n)
        lines.append(f"load {name} data_{name} {fmt([2] * n)}")
        return data["data_" + name]

    def grown(name, first):
        """`first` legs' tensor times one vector of 2^8 values per eight h legs."""
        t, at, vecs = load(name + "0", len(first)), list(first), []
        for i in range(0, nh, 8):
            h = H[i:i + 8]
            vecs.append(load(f"{name}v{i}", len(h)).reshape(-1, order="F"))
            lines.append(f"ncon {name}{i + 8} {fmt(at + h)} {name}{i} {fmt(at)} {name}v{i} {fmt(h)}")
            at += h
        return t, vecs, f"{name}{(nh + 7) // 8 * 8}"

    a, av, an = grown("A", M + K)
    b, bv, bn = grown("B", K + N)
    lines.append(f"ncon C {fmt(N + M + H)} {an} {fmt(M + K + H)} {bn} {fmt(K + N + H)}")
    at, value = N + M + H, 1.0
    for j, i in enumerate(range(0, nh, 8)):
        h = H[i:i + 8]
        w = load(f"W{i}", len(h)).reshape(-1, order="F")
        rest = [x for x in at if x not in h]
        lines.append(f"ncon D{i} {fmt(rest)} {'C' if not j else f'D{i - 8}'} {fmt(at)} W{i} {fmt(h)}")
        at, value = rest, value * np.sum(av[j] * bv[j] * w)
    lines.append(f"save output D{(nh - 1) // 8 * 8}")
    am = a.reshape(2 ** nm, 2 ** nk, order="F")
    bm = b.reshape(2 ** nk, 2 ** nn, order="F")
    return "\n".join(lines) + "\n", data, (value * (am @ bm)).T.reshape(-1, order="F")


def gemm_steps(steps):
    return [s for s in steps if s["variant"].startswith("k_contract_gemm_mfma")]


@pytest.mark.parametrize("nh,nm,nn,nk", [(24, 2, 2, 2), (24, 2, 2, 3), (24, 3, 3, 3), (26, 2, 2, 2), (23, 2, 2, 2),
                                         (22, 2, 2, 2)])
@pytest.mark.parametrize("precision", ["c128", "c64_4m"])
def test_grid_of_many_units_stays_launchable(precision, nh, nm, nn, nk):
    dsl, _, _ = batched_gemm(nh, nm, nn, nk)
    (g,) = [s for s in gemm_steps(_native.inspect(dsl, precision)["steps"]) if s["name"] == "C"]
    assert g["workgroups"] * 256 < 2 ** 32
    assert g["workgroups"] * g["units_per_workgroup"] >= 2 ** nh


@pytest.mark.gpu
@pytest.mark.parametrize("nh,nm,nn,nk,units", [(24, 2, 2, 2, 2), (25, 2, 2, 2, 4), (13, 6, 6, 6, 2), (12, 6, 6, 6, 1)])
def test_workgroups_of_several_units(nh, nm, nn, nk, units):
    """Against the factors' sums.  Each of about forty complex64 roundings on the way is 6e-8
    of its value; the sums over h are of random signs, so errors and values grow alike, and an
    unlucky sum may be a tenth of its usual size: 40 x 6e-8 x 10 = 2.4e-5 of the norm."""
    dsl, data, ref = batched_gemm(nh, nm, nn, nk)
    ex = Executor(dsl, data, precision="c64_4m", batch=1)
    got = np.asarray(ex.amplitudes([""])).reshape(-1)
    (g,) = [s for s in gemm_steps(ex.stats()["batches"][0]["steps"]) if s["name"] == "C"]
    ex.close()
    assert g["units_per_workgroup"] == units
    assert np.linalg.norm(got - ref) <= 2.4e-5 * np.linalg.norm(ref)


# (H, M, N, K bits; operand orders) -> tile: a side of 128 for complex64 in four products, K >= 64,
# from 1024 such tiles
WIDE = [((10, 7, 6, 6), 0, [128, 64, 16]), ((10, 6, 7, 6), 3, [64, 128, 16]), ((9, 7, 7, 6), 5, [128, 64, 16]),
        ((9, 7, 6, 6), 0, [64, 64, 16]), ((10, 7, 6, 5), 0, [64, 64, 16])]


@pytest.mark.gpu
@pytest.mark.parametrize("shape,layout,tile", WIDE)
def test_wide_tiles_are_the_ones_that_run(shape, layout, tile):
    dsl, data, ref = plain_step(41 + layout, *shape, layout & 1, layout >> 1 & 1, layout >> 2)
    ex = Executor(dsl, data, precision="c64_4m", batch=1, kernel=5)
    got = np.asarray(ex.amplitudes([""])).reshape(-1)
    (g,) = gemm_steps(ex.stats()["batches"][0]["steps"])
    ex.close()
    assert sorted(g["tile"]) == sorted(tile)          # (which operand gives the rows is the layout's)
    assert np.linalg.norm(got - ref) <= 5e-6 * np.linalg.norm(ref)

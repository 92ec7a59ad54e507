"""Small steps whose slice-dependent offsets or operands do not fit an item's descriptor run as
launches of their own, and those at the limit as items: four slice terms per operand, 32
variables, operands that reach 2^28 values."""

import itertools

import numpy as np
import pytest

import qxoracle as O
from qxhip import Executor, _native


def terms(n):
    """Two contractions of one level, their operands cut by n variables each."""
    legs = ",".join(["2"] * (n + 1))
    lines = ["# version: 0.4.0", "output O1 1 2"]
    for t in "ABCD":
        lines.append(f"load {t}0 data_{t} {legs}")
        lines += [f"view {t}{j} {t}{j - 1} v{j} {j + 1} 2" for j in range(1, n + 1)]
    own, cut = "{}", ",".join(str(10 + j) for j in range(n))
    lines.append(f"ncon E 1,2 A{n} {own.format(1)},{cut} B{n} {own.format(2)},{cut}")
    lines.append(f"ncon F 2,3 C{n} {own.format(2)},{cut} D{n} {own.format(3)},{cut}")
    lines += ["ncon G 1,3 E 1,2 F 2,3", "ncon H 3 G 1,3 O1 1", "save output H"]
    return "\n".join(lines) + "\n", (2,) * (n + 1)


@pytest.mark.parametrize("n,batched", [(1, True), (4, True), (5, False)])
def test_slice_terms_per_operand(n, batched):
    steps = _native.inspect(terms(n)[0])["steps"]
    assert [s["level"] >= 0 for s in steps if s["name"] in "EF"] == [batched] * 2


@pytest.mark.gpu
@pytest.mark.parametrize("n", [1, 4, 5])
def test_slice_terms_against_the_oracle(n):
    dsl, shape = terms(n)
    rng = np.random.default_rng(n)
    data = {f"data_{t}": rng.normal(size=shape) + 1j * rng.normal(size=shape) for t in "ABCD"}
    ex = Executor(dsl, data, batch=2, fuse_slices=0)
    every = list(O.slice_assignments(O.parse(dsl)))
    for s in range(len(every)):
        ref = np.stack([r.reshape(-1, order="F") for r in O.amplitudes(dsl, data, ["0", "+"], slices=every[s:s + 1])])
        got = np.asarray(ex.amplitudes(["0", "+"], s, s + 1)).reshape(2, -1)
        assert np.max(np.abs(got - ref)) <= 1e-13 * np.max(np.abs(ref)), s
    ex.close()


def many_variables(n):
    """A product of n small contractions over legs that variable j cuts, pairwise joined."""
    lines = ["# version: 0.4.0"]
    for j in range(1, n + 1):
        lines += [f"load A{j} a{j} 2,2", f"load B{j} b{j} 2,2", f"view C{j} A{j} v{j} 2 2", f"view D{j} B{j} v{j} 1 2",
                  f"ncon E{j} 1,3 C{j} 1,2 D{j} 2,3"]
    lines += [f"ncon F{j} 1,3 {'E1' if j == 2 else f'F{j - 1}'} 1,2 E{j} 2,3" for j in range(2, n + 1)]
    return "\n".join(lines + [f"save output F{n}"]) + "\n"


def test_variables_beyond_32_run_on_their_own():
    levels = {s["name"]: s["level"] for s in _native.inspect(many_variables(34))["steps"]}
    for j in range(1, 35):
        assert (levels[f"E{j}"] >= 0) == (j <= 32), j


@pytest.mark.gpu
def test_variables_beyond_32_against_numpy():
    n = 34
    rng = np.random.default_rng(3)
    a, b = (rng.normal(size=(n, 2, 2)) + 1j * rng.normal(size=(n, 2, 2)) for _ in range(2))
    data = {f"a{j + 1}": a[j] for j in range(n)} | {f"b{j + 1}": b[j] for j in range(n)}
    ex = Executor(many_variables(n), data, batch=1)
    for pick in (0, 1, 1 << 31, 1 << 32, 1 << 33, (1 << 34) - 1, 0x2A5A5A5A5):
        got = np.asarray(ex.amplitudes([""], pick, pick + 1)).reshape(2, 2, order="F")
        ref = np.eye(2)
        for j in range(n):
            v = pick >> j & 1
            ref = ref @ np.outer(a[j][:, v], b[j][v])
        assert np.max(np.abs(got - ref)) <= 1e-12 * np.max(np.abs(ref)), pick
    ex.close()


@pytest.mark.parametrize("bits,batched", [(26, True), (27, False), (28, False)])
def test_operands_of_a_long_reach(bits, batched):
    """Views of tensors of 2^(bits + 2) values that leave four of them, 2^(bits + 1) apart."""
    lines = ["# version: 0.4.0"]
    for t in "AB":
        lines += [f"load {t} data_{t} 2,{2 ** bits},2", f"view {t}1 {t} v1 2 {2 ** bits}"]
    for t, q in itertools.product("AB", "CD"):
        lines += [f"load {q}{t} data_{q}{t} 2,2"] if t == "A" else []
    lines += ["ncon E 1,9,4 A1 1,9,3 CA 3,4", "ncon F 5,9,8 B1 5,9,7 DA 7,8", "ncon G 1,4,5,8 E 1,9,4 F 5,9,8",
              "save output G"]
    levels = {s["name"]: s["level"] for s in _native.inspect("\n".join(lines) + "\n")["steps"]}
    assert [(levels[x] >= 0) for x in "EF"] == [batched] * 2

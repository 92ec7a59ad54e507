"""Gradients through a view of an intermediate tensor, in the view's own section and in
another, with the slices contracted inline and looped, against the oracle's amplitudes (which
are linear in each tensor)."""

import numpy as np
import pytest

import qxoracle as O
from qxhip import Executor
from test_inline_slices import data

pytestmark = pytest.mark.gpu

HEAD = """# version: 0.4.0
output O1 1 2
load A data_1 2,2,4
load B data_2 2,4,2
load C data_3 2,2
"""
TAIL = """ncon E 2,5,6 {x} 2,3 B1 5,3,6
ncon F 2,5,7 E 2,5,6 C 6,7
save output F
"""
PROGRAMS = {
    # the viewed tensor depends on the bitstring, as its consumer does
    "same_section": HEAD + "ncon D 2,3 O1 1 A 1,2,3\nview D1 D v1 2 4\nview B1 B v1 2 4\n" + TAIL.format(x="D1"),
    # it does not
    "other_section": HEAD + "load M data_5 4,4\nncon A2 1,2,9 A 1,2,3 M 3,9\nview A1 A2 v1 3 4\nview B1 B v1 2 4\n"
                            "ncon D 2,3 O1 1 A1 1,2,3\n" + TAIL.format(x="D"),
    # a chain of two viewed intermediates
    "two_views": HEAD + "load M data_5 2,2\nncon D 2,3 O1 1 A 1,2,3\nview D1 D v1 2 4\nncon G 8,3 D1 2,3 M 2,8\n"
                        "view G1 G v2 1 2\nload W data_6 2\nview W1 W v2 1 2\nncon K 3 G1 8,3 W1 8\nview B1 B v1 2 4\n"
                        "ncon E 5,6 K 3 B1 5,3,6\nncon F 5,7 E 5,6 C 6,7\nsave output F\n",
}


@pytest.mark.parametrize("options", [{}, {"fuse_slices": 0}, {"graph": 1}, {"batch_last": 1}])
@pytest.mark.parametrize("name", PROGRAMS)
def test_gradient_through_a_viewed_intermediate(name, options):
    dsl, bits = PROGRAMS[name], ["0", "+", "1"]
    values = data(dsl)
    ex = Executor(dsl, values, batch=4, **options)
    rng = np.random.default_rng(1)
    shape = (3, ex.plan.result_elems)
    cot = rng.normal(size=shape) + 1j * rng.normal(size=shape)
    got = ex.vjp(bits, cot)
    ex.close()
    for k, t in values.items():
        ref = np.zeros(t.size, dtype=np.complex128)
        for i in range(t.size):
            unit = np.zeros(t.size, dtype=np.complex128)
            unit[i] = 1
            amps = O.amplitudes(dsl, {**values, k: unit.reshape(t.shape, order="F")}, bits)
            ref[i] = np.sum(cot * np.stack([a.reshape(-1, order="F") for a in amps]).conj())
        assert np.max(np.abs(np.asarray(got[k]).reshape(-1) - ref)) <= 1e-12 * np.max(np.abs(ref)), k

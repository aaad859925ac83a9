"""Three steps a launch (proceed_x3, proceed_adjoint_x3) against three launches of one step, in
a correctly rounded build of the FP32 machine's streaming forms: the same bits on grids whose
strips, rows and chunks end inside the grid, and on boxes smaller than any of them; and the
oracle's bits."""
import numpy as np
import pytest

from helpers import oracle_machine
from paraiso_amd import variants
from paraiso_amd.adjoint import add_adjoint
from paraiso_amd.om.dyn import CType
from paraiso_amd.schemes.linear_wave import linear_wave_om

pytestmark = pytest.mark.gpu
FIELDS = ("fieldF", "fieldG", "adj_fieldF", "adj_fieldG")


def start(n, seed, *machines):
    rng = np.random.default_rng(seed)
    state = [rng.standard_normal(tuple(reversed(n)), dtype=np.float32) for _ in FIELDS]
    for m in machines:
        for k, v in (("c", 1.0), ("dx", 1.0), ("dt", 0.5)):
            m.set(k, v)
        for f, x in zip(FIELDS, state):
            m.set(f, x)


@pytest.mark.parametrize("n", [(3, 5, 4), (4, 5, 3), (61, 6, 17), (64, 4, 9), (58, 8, 4),
                               (125, 9, 33), (70, 33, 21), (200, 130, 100)])
def test_three_steps(require_gpu, n):
    print("wave x3 %s" % (n,), flush=True)
    a, b = (variants.machine("wave3d_f32_precise", n) for _ in range(2))
    start(n, 8, a, b)
    for _ in range(2):
        for kern in ("proceed", "proceed_adjoint"):
            a.run(kern + "_x3")
            for _ in range(3):
                b.run(kern)
    for f in FIELDS:
        assert np.array_equal(a.get(f), b.get(f)), f
    # the same terms, summed in FP64 in another order
    assert abs(a.get("energy") - b.get("energy")) <= 1e-12 * abs(b.get("energy"))


def test_three_steps_are_the_oracles(require_gpu):
    n = (64, 64, 64)
    a = variants.machine("wave3d_f32_precise", n)
    o = oracle_machine(lambda: add_adjoint(linear_wave_om(3, CType.Float), "proceed",
                                           ["fieldF", "fieldG"]), n)
    start(n, 9, a, o)
    print("wave x3 vs the oracle", flush=True)
    a.run("proceed_x3", 3)
    o.run("proceed", 9)
    for f in FIELDS[:2]:
        assert np.array_equal(a.get(f), o.get(f)), f

"""One adjoint step of the FP64 wave takes strips or tiles by the length of the rows and the
number of cells: on both sides of each line the stored bits are those of the machine that has
tiles only."""
import numpy as np
import pytest

from paraiso_amd import variants

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [(255, 7, 6), (256, 7, 6), (257, 5, 9), (70, 240, 238),
                               (70, 241, 240), (63, 280, 230)])
def test_adjoint_step(require_gpu, n):
    print("wave adjoint lines %s" % (n,), flush=True)
    a, b = (variants.machine(v, n) for v in ("wave3d_f64", "wave3d_f64_persist"))
    rng = np.random.default_rng(2)
    state = {f: rng.standard_normal(tuple(reversed(n))) for f in ("adj_fieldF", "adj_fieldG")}
    for m in (a, b):
        for k, v in (("c", 1.0), ("dx", 1.0), ("dt", 0.5)):
            m.set(k, v)
        for f, x in state.items():
            m.set(f, x)
        m.run("proceed_adjoint")
    for f in state:
        assert np.array_equal(a.get(f), b.get(f)), f

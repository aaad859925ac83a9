"""hydro_f32 above the number of cells from which it streams, against the machine that streams at
every size: their kernels are the same plan with its multiply-adds written out, so a cell's bits
do not depend on how the grid was cut into strips and chunks."""
import numpy as np
import pytest

from paraiso_amd import inputs, variants

pytestmark = pytest.mark.gpu
F = ("density", "velocity0", "velocity1", "pressure")


@pytest.mark.parametrize("nx,ny", [(1021, 767), (775, 775), (59, 10240), (10007, 61)])
def test_streaming_steps(require_gpu, nx, ny):
    print("headline lanes %dx%d" % (nx, ny), flush=True)
    a, b = variants.machine("hydro_f32", (nx, ny)), variants.machine("hydro_f32_batch", (nx, ny))
    rng = np.random.default_rng(6)
    state = [(x + 0.1 * rng.standard_normal(x.shape)).astype(np.float32)
             for x in inputs.kh_init(nx, ny, 6)]
    for m in (a, b):
        for k, v in inputs.hydro_scalars(nx, ny).items():
            m.set(k, v)
        for f, x in zip(F, state):
            m.set(f, x)
        m.run("proceed")
        m.run("proceed", 3)
    a.run("proceed_prime")               # in tiles, contracted by the compiler
    b.set("__carry_proceed_0", a.get("__carry_proceed_0"))
    for m in (a, b):
        m.run("proceed_pipelined")
        m.run("proceed_pipelined", 3, graph=True)
    for f in F:
        assert np.array_equal(a.get(f), b.get(f)), f
    assert a.get("time") == b.get("time")

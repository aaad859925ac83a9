"""Runs of calls: pr_run and pr_run_graph make several calls per launch where the machine has a
kernel for it, and leave the scalar stores of Life and LinearWave to the run's end.  Arrays,
counters and reductions are what the same number of single calls leaves."""
import numpy as np
import pytest

from paraiso_amd import inputs, variants

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("count", [1, 2, 3, 4, 7, 8, 9, 12, 31])
@pytest.mark.parametrize("graph", [False, True])
def test_life(require_gpu, count, graph):
    nx, ny = 77, 45
    print("life run of %d, graph %s" % (count, graph), flush=True)
    a, b = variants.machine("life_i32", (nx, ny)), variants.machine("life_i32", (nx, ny))
    for m in (a, b):
        m.run("init")
        m.set("cell", inputs.life_init((ny, nx), 5))
    for _ in range(3):                    # the second graph replay starts on swapped buffers
        a.run("proceed", count, graph=graph)
        for _ in range(count):
            b.run("proceed")
        assert np.array_equal(a.get("cell"), b.get("cell"))
        assert a.get("population") == b.get("population") == int(b.get("cell").sum())
        assert a.get("generation") == b.get("generation")


@pytest.mark.parametrize("count", [1, 2, 5])
def test_wave(require_gpu, count):
    n = (70, 21, 13)
    print("wave run of %d" % count, flush=True)
    a, b = variants.machine("wave3d_f64", n), variants.machine("wave3d_f64", n)
    rng = np.random.default_rng(4)
    state = [rng.standard_normal(tuple(reversed(n))) for _ in range(4)]
    fields = ("fieldF", "fieldG", "adj_fieldF", "adj_fieldG")
    for m in (a, b):
        for k, v in (("c", 1.0), ("dx", 1.0), ("dt", 0.5)):
            m.set(k, v)
        for f, x in zip(fields, state):
            m.set(f, x)
    for graph in (False, True, True):
        for kern in ("proceed", "proceed_adjoint"):
            a.run(kern, count, graph=graph)
            for _ in range(count):
                b.run(kern)
        for f in fields:
            assert np.array_equal(a.get(f), b.get(f)), f
        # the same FP64 terms in another order: 2^-53 a term against a sum of positives
        assert abs(a.get("energy") - b.get("energy")) <= 1e-12 * abs(b.get("energy"))


@pytest.mark.parametrize("count", [1, 2, 3, 4, 7])
def test_wave_large(require_gpu, count):
    """Grids that take three steps a launch (two such launches for three two-step calls)."""
    n = (300, 290, 240)
    print("wave run of %d, %s" % (count, n), flush=True)
    a, b = variants.machine("wave3d_f32", n), variants.machine("wave3d_f32", n)
    rng = np.random.default_rng(5)
    fields = ("fieldF", "fieldG", "adj_fieldF", "adj_fieldG")
    for f in fields:
        x = rng.standard_normal(tuple(reversed(n)), dtype=np.float32)
        a.set(f, x)
        b.set(f, x)
    for m in (a, b):
        for k, v in (("c", 1.0), ("dx", 1.0), ("dt", 0.5)):
            m.set(k, v)
    for kern in ("proceed", "proceed_x2", "proceed_adjoint", "proceed_adjoint_x2"):
        a.run(kern, count)
        for _ in range(count):
            b.run(kern)
    # streamed steps write their multiply-adds out, the same in every kernel; the grid is one
    # that the streaming LDS tiles (contracted by the compiler) do not take
    for f in fields:
        x, y = a.get(f).astype(np.float64), b.get(f)
        assert np.abs(x - y).max() <= 1e-5 * np.abs(y).max(), f
    assert abs(a.get("energy") - b.get("energy")) <= 1e-6 * abs(b.get("energy"))


def test_time_counts_every_call(require_gpu):
    """Hydro at a fixed dt stores its time from scalars alone: n calls add dt n times."""
    nx, ny = 40, 24
    a, b = (variants.machine("hydro_fixed_f64", (nx, ny)) for _ in range(2))
    for m in (a, b):
        for k, v in inputs.hydro_scalars(nx, ny).items():
            m.set(k, v)
        m.set("dt", 1e-4)
        for f, x in zip(("density", "velocity0", "velocity1", "pressure"),
                        inputs.kh_init(nx, ny, 2)):
            m.set(f, x)
    a.run("proceed", 11)
    for _ in range(11):
        b.run("proceed")
    assert a.get("time") == b.get("time")
    assert np.array_equal(a.get("density"), b.get("density"))


@pytest.mark.parametrize("variant,size", [("hydro_f64", (40, 23)), ("hydro_f64", (201, 170)),
                                          ("hydro_f64", (400, 333)), ("hydro_f64", (701, 633)),
                                          ("hydro_f64_lane", (117, 65)),
                                          ("hydro_f32_precise", (130, 67))])
@pytest.mark.parametrize("count,graph", [(2, False), (3, False), (4, True), (5, True)])
def test_hydro_calls_in_one_pass(require_gpu, variant, size, count, graph):
    """A run of ``proceed`` carries its reduction: what single calls leave, and the statics that
    carry it for ``proceed_pipelined`` stay as they were."""
    print("hydro run %s %s of %d, graph %s" % (variant, size, count, graph), flush=True)
    a, b = variants.machine(variant, size), variants.machine(variant, size)
    names = ("density", "velocity0", "velocity1", "pressure")
    rng = np.random.default_rng(8)
    state = [x + 0.05 * rng.standard_normal(x.shape) for x in inputs.kh_init(*size, 6)]
    dt = np.float32 if "f32" in variant else np.float64
    for m in (a, b):
        for k, v in inputs.hydro_scalars(*size).items():
            m.set(k, v)
        for f, x in zip(names, state):
            m.set(f, x.astype(dt))
        m.run("proceed_prime")
    for _ in range(2):
        a.run("proceed", count, graph=graph)
        for _ in range(count):
            b.run("proceed")
        for f in names:
            assert np.array_equal(a.get(f), b.get(f)), f
        for s in ("time", "__carry_proceed_0"):
            assert a.get(s) == b.get(s), s
    for m in (a, b):
        m.run("proceed_pipelined", 3)
    for f in names:
        assert np.array_equal(a.get(f), b.get(f)), f
    assert a.get("time") == b.get("time")

"""Register streaming on the GPU, against the tile forms of the same programs: correctly
rounded builds compute the same operations on the same values, so the stored arrays are the
same bits at every grid size (strips, chunks and rows that end inside the grid, grids smaller
than a strip, and grids shorter than the stencil's reach)."""
import numpy as np
import pytest

from paraiso_amd import inputs, variants

pytestmark = pytest.mark.gpu
F = ("density", "velocity0", "velocity1", "pressure")


def hydro_state(nx, ny, seed):
    rng = np.random.default_rng(seed)
    return [a + 0.1 * rng.standard_normal(a.shape) for a in inputs.kh_init(nx, ny, seed)]


def start(m, nx, ny, seed):
    for k, v in inputs.hydro_scalars(nx, ny).items():
        m.set(k, v)
    for f, a in zip(F, hydro_state(nx, ny, seed)):
        m.set(f, a)


def same(a, b):
    for f in F:
        assert np.array_equal(a.get(f), b.get(f)), f
    assert a.get("time") == b.get("time")


@pytest.mark.parametrize("nx,ny", [(5, 7), (57, 4), (58, 32), (59, 33), (63, 31), (64, 64),
                                   (65, 5), (116, 65), (117, 96), (233, 41)])
def test_hydro_strips_and_chunks(require_gpu, nx, ny):
    print("hydro lane %dx%d" % (nx, ny), flush=True)
    a, b = variants.machine("hydro_f64_lane", (nx, ny)), variants.machine("hydro_f64", (nx, ny))
    for m in (a, b):
        start(m, nx, ny, 3)
        m.run("proceed", 2)
        m.run("proceed_prime")
        m.run("proceed_pipelined", 3)
    same(a, b)


def test_hydro_on_both_sides_of_the_rule(require_gpu):
    """hydro_f64 takes the tile form below its smallest streaming grid and streams above it:
    both against the machine that streams LDS tiles."""
    for nx, ny in ((640, 600), (701, 633)):
        print("hydro rule %dx%d" % (nx, ny), flush=True)
        a, b = variants.machine("hydro_f64", (nx, ny)), variants.machine("hydro_f64_march", (nx, ny))
        for m in (a, b):
            start(m, nx, ny, 5)
            m.run("proceed_prime")
            m.run("proceed_pipelined", 2)
            m.run("proceed", 1)
        same(a, b)


@pytest.mark.parametrize("batch", [False, True])
def test_hydro_rows_past_32_bit_offsets(require_gpu, batch):
    """A row of 2^29 cells or more takes the kernels with 64-bit lane offsets: one row of a
    repeated pattern (its period divides the row), against the small grid of one period."""
    period, times = 8191, 65545
    nx = period * times
    print("hydro lane far rows %d" % nx, flush=True)
    b = variants.batch("hydro_f64_lane", [(nx, 1)]) if batch else None
    m = b.grids[0] if batch else variants.machine("hydro_f64_lane", (nx, 1))
    one = variants.machine("hydro_f64", (period, 1))
    for k, v in inputs.hydro_scalars(period, 1).items():
        m.set(k, v)
        one.set(k, v)
    for f, a in zip(F, hydro_state(period, 1, 9)):
        one.set(f, a)
        m.set(f, np.tile(a.reshape(1, -1), (1, times)))
    (b or m).run("proceed")
    one.run("proceed")
    for f in F:
        got = m.get(f).reshape(times, period)
        assert (got == one.get(f).reshape(1, -1)).all(), f
        print("same", f, flush=True)


@pytest.mark.parametrize("count,lo,hi", [(5, 5, 90), (9, 64, 700)])
def test_hydro_batch(require_gpu, count, lo, hi):
    """Few tiles are split over a workgroup's waves, many are a wave's each."""
    sizes = [tuple(int(v) for v in s) for s in inputs.batched_sizes(count, 11, lo, hi)]
    print("hydro lane batch", sizes, flush=True)
    b = variants.batch("hydro_f64_lane", sizes)
    ms = [variants.machine("hydro_f64", s) for s in sizes]
    for g, (nx, ny) in enumerate(sizes):
        for m in (b.grids[g], ms[g]):
            start(m, nx, ny, g)
    b.run("proceed_prime")
    b.run("proceed_pipelined", 3, graph=True)
    b.run("proceed", 1)
    b.sync()
    for g, m in enumerate(ms):
        m.run("proceed_prime")
        m.run("proceed_pipelined", 3)
        m.run("proceed", 1)
        same(b.grids[g], m)


@pytest.mark.parametrize("n", [(4, 5, 3), (64, 4, 9), (61, 6, 17), (62, 8, 4), (125, 9, 33),
                               (70, 33, 21)])
def test_wave_rows_strips_and_chunks(require_gpu, n):
    print("wave lane %s" % (n,), flush=True)
    a, b = (variants.machine(v, n) for v in ("wave3d_f64", "wave3d_f64_persist"))
    rng = np.random.default_rng(8)
    state = {f: rng.standard_normal(tuple(reversed(n)))
             for f in ("fieldF", "fieldG", "adj_fieldF", "adj_fieldG")}
    for m in (a, b):
        for k, v in (("c", 1.0), ("dx", 1.0), ("dt", 0.5)):
            m.set(k, v)
        for f, x in state.items():
            m.set(f, x)
        for kern in ("proceed", "proceed_adjoint"):
            m.run(kern, 2)
        if min(n) >= 4:
            for kern in ("proceed_x2", "proceed_adjoint_x2"):
                m.run(kern, 2)
    for f in state:
        assert np.array_equal(a.get(f), b.get(f)), f
    # the same FP64 terms summed in another order: 2^-53 a term against a sum of positives
    assert abs(a.get("energy") - b.get("energy")) <= 1e-12 * abs(b.get("energy"))

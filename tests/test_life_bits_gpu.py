"""Life in bit planes against a numpy brute force: squares, strips and chunks that end inside
the grid, grids smaller than a square and than the stencil's reach, and cells that hold other
numbers than 0 and 1 (a wave that reads one computes its square by streaming)."""
import numpy as np
import pytest

from paraiso_amd import inputs, variants

pytestmark = pytest.mark.gpu


def generation(c):
    n = sum(np.roll(c, (a, b), (0, 1)) for a in (-1, 0, 1) for b in (-1, 0, 1)) - c
    return (((c == 0) & (n == 3)) | ((c == 1) & (n >= 2) & (n <= 3))).astype(np.int32)


@pytest.mark.parametrize("nx,ny", [(3, 5), (17, 40), (32, 32), (33, 31), (48, 96), (56, 57),
                                   (64, 64), (65, 129), (200, 50)])
@pytest.mark.parametrize("kernel,n", [("proceed_x4", 4), ("proceed_x8", 8), ("proceed_x16", 16)])
@pytest.mark.parametrize("other", [False, True])
def test_squares(require_gpu, nx, ny, kernel, n, other):
    print("life bits %dx%d %s other %s" % (nx, ny, kernel, other), flush=True)
    cell = inputs.life_init((ny, nx), 7)
    if other:
        cell[ny // 2, nx // 3], cell[0, 0], cell[-1, -1] = 2, -1, 1 << 30
    m = variants.machine("life_i32", (nx, ny))
    m.run("init")
    m.set("cell", cell)
    m.run(kernel)
    for _ in range(n):
        cell = generation(cell)
    assert np.array_equal(m.get("cell"), cell)
    assert m.get("population") == int(cell.sum()) and m.get("generation") == n


@pytest.mark.parametrize("other", [False, True])
def test_one_generation_of_a_large_grid(require_gpu, other):
    nx, ny = 1250, 811
    print("life bits %dx%d proceed other %s" % (nx, ny, other), flush=True)
    cell = inputs.life_init((ny, nx), 9)
    if other:
        cell[100, 700], cell[810, 0] = 3, -2
    m = variants.machine("life_i32", (nx, ny))
    m.run("init")
    m.set("cell", cell)
    m.run("proceed")
    cell = generation(cell)
    assert np.array_equal(m.get("cell"), cell)
    assert m.get("population") == int(cell.sum())

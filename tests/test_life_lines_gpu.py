"""The launch form of Life's kernels depends on the number of cells: on both sides of each line,
against the numpy brute force."""
import numpy as np
import pytest

from paraiso_amd import inputs, variants
from test_life_bits_gpu import generation

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kernel,n,nx,ny", [("proceed", 1, 1090, 1100), ("proceed", 1, 1100, 1091),
                                            ("proceed", 1, 40, 30001), ("proceed_x4", 4, 640, 624),
                                            ("proceed_x4", 4, 640, 625), ("proceed_x4", 4, 50, 8003)])
@pytest.mark.parametrize("other", [False, True])
def test_both_sides(require_gpu, kernel, n, nx, ny, other):
    print("life lines %s %dx%d other %s" % (kernel, nx, ny, other), flush=True)
    cell = inputs.life_init((ny, nx), 4)
    if other:
        cell[ny // 3, nx // 2], cell[-1, 0] = 5, -7
    m = variants.machine("life_i32", (nx, ny))
    m.run("init")
    m.set("cell", cell)
    m.run(kernel)
    for _ in range(n):
        cell = generation(cell)
    assert np.array_equal(m.get("cell"), cell)
    assert m.get("population") == int(cell.sum()) and m.get("generation") == n

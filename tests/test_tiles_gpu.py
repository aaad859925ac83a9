"""The tile a launch takes depends on the grid's size: on both sides of every line, and on
grids too thin for the small tiles' partials, the stored bits are those of the machine that
streams at every size."""
import numpy as np
import pytest

from paraiso_amd import variants
from test_lane_gpu import same, start

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nx,ny", [(3, 4), (15, 9), (17, 8), (200, 149), (201, 150), (1, 29999),
                                   (29999, 1), (400, 299), (401, 300), (7, 17000)])
def test_hydro_tiles(require_gpu, nx, ny):
    print("hydro tiles %dx%d" % (nx, ny), flush=True)
    a, b = variants.machine("hydro_f64", (nx, ny)), variants.machine("hydro_f64_lane", (nx, ny))
    for m in (a, b):
        start(m, nx, ny, 6)
        m.run("proceed", 2)
        m.run("proceed_prime")
        m.run("proceed_pipelined", 2)
    same(a, b)

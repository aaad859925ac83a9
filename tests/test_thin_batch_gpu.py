"""Batches of long thin grids, above the number of cells from which a single grid streams: the
batch's LDS tiles wrap several times around the short axis.  The stored bits are those of the
machine that streams at every size."""
import pytest

from paraiso_amd import variants
from test_lane_gpu import same, start

pytestmark = pytest.mark.gpu
THIN = (2, 3, 7, 10, 17, 24, 33, 40)


def test_thin_grids(require_gpu):
    sizes = [(410_000 // n + 1, n) for n in THIN] + [(n, 410_000 // n + 1) for n in THIN]
    b = variants.batch("hydro_f64", sizes)
    for g, (nx, ny) in enumerate(sizes):
        start(b.grids[g], nx, ny, g)
    b.run("proceed")
    b.run("proceed_prime")
    b.run("proceed_pipelined", 2)
    b.sync()
    for g, (nx, ny) in enumerate(sizes):
        print("thin grid %dx%d" % (nx, ny), flush=True)
        m = variants.machine("hydro_f64_lane", (nx, ny))
        start(m, nx, ny, g)
        m.run("proceed")
        m.run("proceed_prime")
        m.run("proceed_pipelined", 2)
        same(b.grids[g], m)
        m.close()

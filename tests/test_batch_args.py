"""The packed arguments of a batch's grids (no GPU call is made): a batch runs the launch's LDS
tiles whatever form a single grid of the size would take, so its ``wide`` flag has to cover
those tiles: where it is 0, om_wrap adds or takes the extent off once, which must leave every
coordinate that a tile reads inside the grid."""
import ctypes
import re

import pytest

from paraiso_amd import variants
from paraiso_amd.generator import _hip_sources
from paraiso_amd.generator.hip.ir import lower_kernel
from paraiso_amd.generator.hip.schedule import lds_budget, schedule_kernel
from paraiso_amd.generator.plan import translate
from paraiso_amd.machine import PrMachineDesc

P, I, U = ctypes.c_void_p, ctypes.c_int, ctypes.c_uint


class Ctx(ctypes.Structure):
    _fields_ = [("cur", P), ("next", P), ("scal", P), ("part", P), ("counter", P), ("n", I * 3),
                ("tiles", I * 3), ("ntiles", U), ("stream", P), ("run", P), ("fold", P)]


def args_type(src, fn):
    """The struct Args_<fn> of the generated source as a ctypes structure."""
    at = src.index("struct Args_%s {" % fn)
    fields = []
    for line in re.sub(r"/\*.*?\*/", "", src[at:src.index("};", at)], flags=re.S).split("\n")[1:]:
        for part in line.split(";"):
            if part.strip():
                t = P if "*" in part else U if part.split()[0] == "unsigned" else I
                names = re.sub(r"^.*\*|__restrict__", "", part) if t is P else \
                    part.split(None, 1)[1]
                fields += [(x.strip(), t) for x in names.split(",")]
    return type("Args", (ctypes.Structure,), {"_fields_": fields})


def halos(name):
    """Largest offset each launch of the variant's kernels reads at, by kernel and launch."""
    mk, _, precise = variants.VARIANTS[name]
    setup = variants.setup_of(name)
    om = translate(setup, mk()).om
    out = {}
    for ki, k in enumerate(om.kernels):
        f = setup.form_of(k.name)
        sch = schedule_kernel(lower_kernel(om, ki, (True, True), exact=not precise), f["tile"],
                              lds_budget(f["threads"]), f["mat_gain"])
        out[k.name] = [max([0] + [max(-lo, hi) for ph in la.phases for lo, hi in ph.box])
                       for la in sch.launches]
    return out


@pytest.mark.parametrize("name", ["hydro_f32", "hydro_f64"])
def test_wide_covers_the_tiles(name):
    mk, _, precise = variants.VARIANTS[name]
    src = _hip_sources(variants.setup_of(name), mk(), precise)[1]
    lib = ctypes.CDLL(variants.library(name))
    lib.pm_describe.restype = ctypes.POINTER(PrMachineDesc)
    d = lib.pm_describe().contents
    nothing = (P * d.n_static)()
    reach = halos(name)
    thin = list(range(1, 49)) + [63, 64, 65]
    sizes = [(-(-700_000 // t), t) for t in thin] + [(t, -(-700_000 // t)) for t in thin]
    sizes += [(t, 40) for t in thin] + [(1021, 767), (2048, 2048)]
    seen = 0
    for ki in range(d.n_kernel):
        k = d.kernels[ki]
        for li in range(k.n_launch):
            la = k.launches[li]
            if not la.tile[0]:
                continue
            Args = args_type(src, "Hydro_%s_l%d" % (k.name.decode(), li))
            assert ctypes.sizeof(Args) == la.args_size
            pack = ctypes.CFUNCTYPE(None, ctypes.POINTER(Ctx), ctypes.POINTER(Args))(la.pack)
            h = reach[k.name.decode()][li]
            for size in sizes:
                n = tuple(size) + (1,)
                tiles = [-(-n[ax] // la.tile[ax]) for ax in range(3)]
                c = Ctx(cur=ctypes.cast(nothing, P), next=ctypes.cast(nothing, P), n=(I * 3)(*n),
                        tiles=(I * 3)(*tiles), ntiles=tiles[0] * tiles[1] * tiles[2])
                a = Args()
                pack(ctypes.byref(c), ctypes.byref(a))
                assert (a.n0, a.n1, a.ntiles) == (n[0], n[1], c.ntiles)
                for ax in range(2):
                    lo, hi = -h, (tiles[ax] - 1) * la.tile[ax] + la.tile[ax] - 1 + h
                    if lo < -n[ax] or hi >= 2 * n[ax]:
                        assert a.wide, (k.name, li, size, "reads %d..%d" % (lo, hi))
                        seen += 1
    assert seen > 20

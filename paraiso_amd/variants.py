"""The machines this package builds ahead of time, one shared library each.

Grid sizes are run-time parameters of a machine, so one library serves every
size of its program.  The ratio of specific heats and the dt mode are baked
into the OM of a Hydro program, as in the reference.
"""
from __future__ import annotations

from fractions import Fraction

from . import annotation as A
from .generator import Language, Setup, build_machine
from .om.dyn import CType

CYC2 = (A.Condition.Cyclic,) * 2
CYC3 = (A.Condition.Cyclic,) * 3
CYC1 = (A.Condition.Cyclic,)
OPEN2 = (A.Condition.Open,) * 2


def _life():
    """Life with ``proceed_x4``, ``proceed_x8`` and ``proceed_x16``: four, eight or sixteen
    generations per launch (temporal blocking)."""
    from .schemes.life import life_om
    from .transform import unroll
    return unroll(unroll(unroll(life_om(), "proceed", 4), "proceed", 8), "proceed", 16)


def _life_plain():
    from .schemes.life import life_om
    return life_om()


def _life_legacy():
    from .schemes.life import life_om_legacy
    return life_om_legacy()


def _hydro_legacy():
    from .schemes.hydro import hydro_om_legacy
    return hydro_om_legacy()


def _hydro(real, gamma=Fraction(7, 5), dt_mode="cfl"):
    """Hydro with, beside ``proceed``, ``proceed_prime`` + ``proceed_pipelined``: the CFL
    minimum of the next step computed in the store phase of this one (one grid pass)."""
    def mk():
        from .schemes.hydro import hydro_om
        from .transform import pipeline_reduce
        om = hydro_om(real, gamma, dt_mode)
        return pipeline_reduce(om, "proceed") if dt_mode == "cfl" else om
    return mk


def _wave(ndim=3, real=CType.Float):
    def mk():
        from .schemes.linear_wave import linear_wave_om
        return linear_wave_om(ndim, real)
    return mk


HYDRO_FIELDS = ["density", "velocity0", "velocity1", "pressure"]


def _hydro_adj(real):
    def mk():
        from .adjoint import add_adjoint
        from .schemes.hydro import hydro_om
        return add_adjoint(hydro_om(real, Fraction(7, 5), "fixed"), "proceed", HYDRO_FIELDS)
    return mk


STAGE_FIELDS = ["stage_" + f for f in HYDRO_FIELDS]


def _hydro_adj_staged(real):
    """The fixed-dt step split into its two stages (``proceed_stage1`` stores the half-step
    state, ``proceed_stage2`` finishes the step from it), with one adjoint kernel per stage:
    the checkpoint driver replays both stages and runs ``proceed_stage2_adjoint`` then
    ``proceed_stage1_adjoint``, so no adjoint launch recomputes stage 1 under the halo that
    stage 2 needs."""
    def mk():
        from .adjoint import add_adjoint
        from .schemes.hydro import hydro_om
        om = hydro_om(real, Fraction(7, 5), "fixed", stages=True)
        om = add_adjoint(om, "proceed_stage2", HYDRO_FIELDS + STAGE_FIELDS,
                         zero_in=STAGE_FIELDS)
        return add_adjoint(om, "proceed_stage1", HYDRO_FIELDS + STAGE_FIELDS)
    return mk


def _wave_adj(ndim, real, most=2):
    """LinearWave with its adjoint, and both fused two steps per launch (``proceed_x2``,
    ``proceed_adjoint_x2``), or up to ``most``."""
    def mk():
        from .adjoint import add_adjoint
        from .schemes.linear_wave import linear_wave_om
        from .transform import unroll
        om = add_adjoint(linear_wave_om(ndim, real), "proceed", ["fieldF", "fieldG"])
        for k in range(2, most + 1):
            om = unroll(unroll(om, "proceed", k), "proceed_adjoint", k)
        return om
    return mk


def _optable(real):
    def mk():
        from .schemes.optable import optable_om
        return optable_om(real)
    return mk


def _rewrites():
    from .schemes.rewrites import rewrites_om
    return rewrites_om()


def _monitor():
    from .schemes.monitor import monitor_om
    return monitor_om()


def _monitor_fused():
    """With ``watch_x2`` and ``watch_x4``."""
    from .transform import unroll
    return unroll(unroll(_monitor(), "watch", 2), "watch", 4)


# Register streaming (generator/hip/lane.py).  Hydro: a wave streams along y; below min_cells
# the strips are too short for their run-up and the tile form is faster (FP32: 22.6 us a step
# at 700^2 in tiles, 24.0 streaming; 33.4 and 28.3 at 1021x767; 112 and 91 at 2048^2.  FP64:
# 31.9 and 33.7 at 512^2, 55.9 and 51.2 at 700^2, 344 and 250 at 2048^2).
LANE_HYDRO_F32 = {"waves": 4, "occupancy": 2, "steps": 4, "min_cells": 600_000}
LANE_HYDRO_F64 = {"waves": 4, "occupancy": 2, "steps": 4, "min_cells": 400_000}
# Below that, tiles by the number of cells: a small grid is a matter of how long a workgroup
# takes, which small tiles with one loop point per work-item and phase shorten.  FP32, us a
# step at 96x64, 400x300, 512^2, 700^2: 16x8 tiles 7.7 13.7 20.1 30.2, 32x16 10.6 12.2 14.4
# 21.7, 64x32 resident 17.8 18.5 18.7 22.3.  FP64 at 96x64, 300x200, 512^2: 16x8 11.5 21.2 64,
# 16x16 13.4 15.4 43.6, 32x32 resident 26.9 28.0 31.7.
TINY_HYDRO_F32 = ({"below": 60_000, "tile": (16, 8), "threads": 320},)
TINY_HYDRO_F64 = ({"below": 30_000, "tile": (16, 8), "threads": 320},
                  {"below": 120_000, "tile": (16, 16), "threads": 512})
# The pass that only reduces (``proceed_prime``) reads each cell once and keeps the tiles: us a
# call in strips and in 64x32 tiles, FP32 at 2048^2 17.3 and 13.8, FP64 (32x32) 20x30000 11.4 and
# 8.6.
PRIME_HYDRO_F32 = (("proceed_prime", {"lane": None, "tiny": (), "tile": (64, 32), "threads": 1024,
                                      "mat_gain": 48, "persist": True}),)
PRIME_HYDRO_F64 = (("proceed_prime", {"lane": None, "tiny": ()}),)
# Batches: a tile is 24 steps of one wave: 256 uneven grids 0.92 ms a step in LDS tiles, 0.58 so
# (32 steps: 0.59; small batches 18.5 us a step against 17.6).
# A grid of its own takes fewer steps a wave: us a step of 24, 4 and 2 at 64x48, 400x300 and 700^2
# 36 37 39, 12.2 13.7 21.3, 11.0 13.2 21.5 (LDS tiles 11.7 12.6 22.1).
LANE_HYDRO_BATCH = {"waves": 4, "occupancy": 2, "steps": 24, "least": 2, "always": True}
# LinearWave 3-D: a lane holds rows of y, fewer on small grids (64^3: 11.6 us a step with 8, 8.9
# with 4; 128^3 15.3 and 13.9; 300^3 128 and 128, two steps 123 and 141).  FP32 keeps its
# streaming tiles where they fill the chip: at 512^3 they move 4.7 TB/s and the waves' unaligned
# rows 3.6 (``ratio``), but a 201x150x97 box is 40 tiles (172 us a step) and 1,500 waves (18 us),
# 192^3 148 and 27 us.  FP64: 51 us in tiles and 32 streaming at 160^3, 327 and 220 at 300^3,
# three rows a lane at 100x150x80 15.6 us, four 17.1.
LANE_WAVE_F32 = {"rows": 8, "waves": 4, "occupancy": 3, "steps": 4, "fill": 3, "ratio": 0.75,
                 "small": {"rows": 4, "occupancy": 4, "fill": 4, "below": 2_500_000}}
LANE_WAVE_F64 = {"rows": 4, "waves": 4, "occupancy": 2, "steps": 4, "fill": 3,
                 "small": {"rows": 3, "occupancy": 3, "below": 2_000_000}}
# One adjoint step reads and writes two fields and computes little: tiles, whose rows are aligned,
# are as fast or faster on long rows and large grids.  us a call in strips and in tiles: 512^3
# 1060 and 960, 200^3 50.7 and 44.0, 500x8x500 17.2 and 12.9, 201x150x97 16.2 and 19.9, 150^3 23.4
# and 28.6, 8x500x500 39 and 79.
WAVE_F64_FORMS = (("proceed_adjoint", {"lane": dict(LANE_WAVE_F64, rows_below=256,
                                                    cells_below=4_000_000)}),)

# Life in bit planes (generator/hip/bits.py): 1024^2, 16 generations 7.1 us a launch (the LDS
# tiles took 10 us for eight), 4096^2 eight 31 us against 162 (4.4 TB/s).  Few generations a
# launch are a matter of latency on small grids, where the tiles are faster: us a call of one
# generation in tiles and bits 6.8 and 9.4 at 1024^2, 10.3 and 9.5 at 1200^2, 12.8 and 9.3 at
# 1448^2; of four 7.6 and 9.6 at 512^2, 10.7 and 9.6 at 724^2; of eight 10.5 and 8.7 at 64^2.
BITS = {"bits": True, "waves": 4, "occupancy": 4, "steps": 8}
LIFE_FORMS = (("proceed", {"lane": dict(BITS, min_cells=1_200_000)}),
              ("proceed_x4", {"lane": dict(BITS, min_cells=400_000)}), ("proceed_x8", {"lane": BITS}),
              ("proceed_x16", {"lane": BITS}))

# Runs of calls take the kernels that make several at once (transform.unroll).
FUSED_LIFE = (("proceed", "proceed_x4", 4, 1, 0), ("proceed", "proceed_x8", 8, 1, 0),
              ("proceed", "proceed_x16", 16, 1, 0), ("proceed_x8", "proceed_x16", 2, 1, 0),
              ("proceed_x4", "proceed_x16", 4, 1, 0), ("proceed_x4", "proceed_x8", 2, 1, 0))
FUSED_WAVE = (("proceed", "proceed_x2", 2, 1, 0), ("proceed_adjoint", "proceed_adjoint_x2", 2, 1, 0))
# Three steps a launch pay where memory bounds: 512^3 212 us a step (two: 262), 192^3 17 (16).
LARGE = 20_000_000
FUSED_WAVE_F32 = FUSED_WAVE + tuple(
    (k + x, k + "_x3", n, times, LARGE) for k in ("proceed", "proceed_adjoint")
    for x, n, times in (("", 3, 1), ("_x2", 3, 2)))
THREE = {"lane": {"rows": 8, "waves": 4, "occupancy": 2, "steps": 4, "fill": 2}}
WAVE_FORMS = (("proceed_x3", THREE), ("proceed_adjoint_x3", THREE))

# name -> (OM factory, setup, precise)
VARIANTS = {
    "life_i32": (_life, Setup((64, 64), Language.HIP, boundary=CYC2, fused=FUSED_LIFE,
                              kernel_forms=LIFE_FORMS), True),
    "hydro_f32": (_hydro(CType.Float), Setup((64, 64), Language.HIP, boundary=CYC2, batched=True,
                                             lane=LANE_HYDRO_F32, tiny=TINY_HYDRO_F32,
                                             kernel_forms=PRIME_HYDRO_F32), False),
    # the FP32 step in 64x32 LDS tiles with the resident tile loop, correctly rounded: checked
    # bit for bit against the oracle (the headline machine streams; hydro_f64_lane is its
    # streaming form's bit-for-bit check)
    "hydro_f32_precise": (_hydro(CType.Float), Setup((64, 64), Language.HIP, boundary=CYC2,
                                                     tile=(64, 32), threads=1024, persist=True),
                          True),
    # the same machine, tuned for batches of small uneven grids
    "hydro_f32_batch": (_hydro(CType.Float), Setup((64, 64), Language.HIP, boundary=CYC2,
                                                   batched=True, lane=LANE_HYDRO_BATCH), False),
    "hydro_f64": (_hydro(CType.Double), Setup((64, 64), Language.HIP, boundary=CYC2, batched=True,
                                              lane=LANE_HYDRO_F64, tiny=TINY_HYDRO_F64,
                                              kernel_forms=PRIME_HYDRO_F64), True),
    # register streaming at every size, correctly rounded: checked bit for bit
    "hydro_f64_lane": (_hydro(CType.Double), Setup((64, 64), Language.HIP, boundary=CYC2,
                                                   batched=True, lane=LANE_HYDRO_BATCH), True),
    "hydro_adj_f32": (_hydro_adj(CType.Float), Setup((64, 64), Language.HIP, boundary=CYC2,
                                                     tile=(32, 8)), True),
    # FP32 bulk arithmetic with the hardware reciprocal and square root in the adjoint too
    "hydro_adj_f32_fast": (_hydro_adj(CType.Float), Setup((64, 64), Language.HIP, boundary=CYC2,
                                                          tile=(32, 8), merge_selects=False),
                           False),
    # the fixed-dt step in FP32 (fast arithmetic): streaming like the headline on large grids, in
    # 64x32 tiles with the resident tile loop on small ones
    "hydro_fixed_f32": (_hydro(CType.Float, dt_mode="fixed"),
                        Setup((64, 64), Language.HIP, boundary=CYC2, tile=(64, 32), threads=1024,
                              persist=True, lane=LANE_HYDRO_F32), False),
    # the plain FP64 fixed-dt step at its fastest launch form (the comparison for the adjoint)
    "hydro_fixed_f64": (_hydro(CType.Double, dt_mode="fixed"),
                        Setup((64, 64), Language.HIP, boundary=CYC2, tile=(32, 32), threads=1024,
                              persist=True, lane=LANE_HYDRO_F64), True),
    "hydro_adj_f64": (_hydro_adj(CType.Double), Setup((64, 64), Language.HIP, boundary=CYC2,
                                                      tile=(32, 8)), True),
    # the adjoint per stage (see _hydro_adj_staged), FP32 fast and FP64 correctly rounded
    "hydro_adj2_f32_fast": (_hydro_adj_staged(CType.Float),
                            Setup((64, 64), Language.HIP, boundary=CYC2, tile=(32, 8),
                                  merge_selects=False), False),
    "hydro_adj2_f64": (_hydro_adj_staged(CType.Double),
                       Setup((64, 64), Language.HIP, boundary=CYC2, tile=(32, 8)), True),
    # the same with the adjoint kernels' shared expansions joined into earlier phases
    # (correctly rounded, so bit-identical to the above)
    "hydro_adj2_f64_join": (_hydro_adj_staged(CType.Double),
                            Setup((64, 64), Language.HIP, boundary=CYC2, tile=(32, 16),
                                  threads=512,
                                  kernel_forms=(("proceed_stage1_adjoint", {"join": True}),
                                                ("proceed_stage2_adjoint", {"join": True}))),
                            True),
    "wave3d_f32": (_wave_adj(3, CType.Float, 3), Setup((64, 64, 64), Language.HIP, boundary=CYC3,
                                                    lane=LANE_WAVE_F32, fused=FUSED_WAVE_F32,
                                                    kernel_forms=WAVE_FORMS), False),
    "wave3d_f64": (_wave_adj(3, CType.Double), Setup((64, 64, 64), Language.HIP, boundary=CYC3,
                                                     lane=LANE_WAVE_F64, fused=FUSED_WAVE,
                                                     kernel_forms=WAVE_F64_FORMS), True),
    # the FP32 machine's streaming forms, correctly rounded: checked bit for bit
    "wave3d_f32_precise": (_wave_adj(3, CType.Float, 3), Setup((64, 64, 64), Language.HIP,
                                                            boundary=CYC3, lane=LANE_WAVE_F32,
                                                            kernel_forms=WAVE_FORMS), True),
    # streaming along the last axis (rings of planes in LDS), checked bit for bit
    "life_i32_march": (_life, Setup((64, 64), Language.HIP, boundary=CYC2, tile=(64, 32),
                                    march=4, fused=FUSED_LIFE), True),
    "hydro_f64_march": (_hydro(CType.Double), Setup((64, 64), Language.HIP, boundary=CYC2,
                                                    tile=(64, 32), march=4), True),
    # a tile whose load and annotated-value tiles alone overflow LDS: the scheduler reads the
    # loads from memory and evaluates some annotated values in registers, checked bit for bit
    "hydro_f64_shed": (_hydro(CType.Double), Setup((64, 64), Language.HIP, boundary=CYC2,
                                                   tile=(64, 32), threads=1024), True),
    "wave3d_f64_march": (_wave_adj(3, CType.Double), Setup((64, 64, 64), Language.HIP,
                                                           boundary=CYC3, tile=(32, 8, 32),
                                                           march=1), True),
    # the reference's own LinearWave is 1-D (Convergence.hs:25-54): 1-D and 2-D machines of
    # the same program, checked bit for bit
    "wave1d_f64": (_wave_adj(1, CType.Double), Setup((256,), Language.HIP, boundary=CYC1,
                                                     tile=(256,), threads=256), True),
    "wave2d_f64": (_wave_adj(2, CType.Double), Setup((64, 64), Language.HIP, boundary=CYC2,
                                                     tile=(32, 16), threads=512), True),
    # block tiles with the resident tile loop, whose load phase computes the half step f1
    # from the next tile's prefetched fields, checked bit for bit
    "wave3d_f64_persist": (_wave_adj(3, CType.Double), Setup((64, 64, 64), Language.HIP,
                                                             boundary=CYC3, tile=(16, 8, 8),
                                                             threads=512, persist=True), True),
    # every operator the emitters lower, one per static (checked against the oracle)
    "optable_f32": (_optable(CType.Float), Setup((64, 48), Language.HIP, boundary=CYC2), True),
    "optable_f32_fast": (_optable(CType.Float), Setup((64, 48), Language.HIP, boundary=CYC2),
                         False),
    "optable_f64": (_optable(CType.Double), Setup((64, 48), Language.HIP, boundary=CYC2), True),
    "optable_i32": (_optable(CType.Int), Setup((64, 48), Language.HIP, boundary=CYC2), True),
    # what fast FP32 streaming evaluates in another form (schemes/rewrites.py), streaming and in
    # tiles
    "rewrites_f32": (_rewrites, Setup((64, 64), Language.HIP, boundary=CYC2,
                                      lane=LANE_HYDRO_BATCH), False),
    "rewrites_f32_tiles": (_rewrites, Setup((64, 64), Language.HIP, boundary=CYC2, tile=(32, 8)),
                           False),
    # scalar statics of every kind of dependence on reductions and calls (schemes/monitor.py),
    # in LDS tiles
    "monitor_f64": (_monitor, Setup((64, 64), Language.HIP, boundary=CYC2, tile=(32, 8)), True),
    # the same in batches that stream tiles of ten steps, shared by workgroups of four waves, and
    # with kernels that make two and four calls, the four by way of the two
    "monitor_f64_batch": (_monitor_fused,
                          Setup((64, 64), Language.HIP, boundary=CYC2, batched=True,
                                lane=dict(LANE_HYDRO_BATCH, steps=10),
                                fused=(("watch", "watch_x2", 2, 1, 0),
                                       ("watch_x2", "watch_x4", 2, 1, 0))), True),
    # Open (non-periodic) boundaries: ghost margins, as the reference's shipped examples
    "life_open_i32": (_life_plain, Setup((128, 128), Language.HIP, boundary=OPEN2), True),
    "life_legacy_open_i32": (_life_legacy, Setup((128, 128), Language.HIP, boundary=OPEN2), True),
    "hydro_legacy_open_f32": (_hydro_legacy, Setup((1024, 1024), Language.HIP, boundary=OPEN2),
                              True),
}


def setup_of(name: str):
    """The variant's setup, with the tile the autotuner recorded (paraiso_amd/tuned.json)."""
    from .autotune import tuned
    mk, setup, precise = VARIANTS[name]
    rec = tuned().get(name)
    if rec is not None and "tile" in rec:
        setup = setup.with_(tile=tuple(rec["tile"]), threads=int(rec.get("threads", 256)),
                            mat_gain=int(rec.get("mat_gain", 48)), march=int(rec.get("march", 0)),
                            persist=bool(rec.get("persist", setup.persist)),
                            join=bool(rec.get("join", setup.join)))
    if rec is not None and "kernel_forms" in rec:
        # (over the variant's own forms: a recorded tile keeps a kernel's streaming form)
        forms = dict(setup.kernel_forms)
        for k, f in sorted(rec["kernel_forms"].items()):
            form = dict(forms.get(k, {}))
            if "tile" in f:
                form.update({"tile": tuple(f["tile"]), "threads": int(f["threads"]),
                             "mat_gain": int(f.get("mat_gain", 48)),
                             "march": int(f.get("march", 0)),
                             "persist": bool(f.get("persist", False)),
                             "join": bool(f.get("join", False))})
            # the per-node Manifest/Delayed choices the autotuner kept
            for key in ("manifest", "delayed"):
                if f.get(key):
                    form[key] = tuple(int(v) for v in f[key])
            forms[k] = form
        setup = setup.with_(kernel_forms=tuple(sorted(forms.items())))
    return setup


def build(name: str, force: bool = False) -> str:
    mk, _, precise = VARIANTS[name]
    return build_machine(setup_of(name), mk(), name, precise=precise, force=force)


def build_all(force: bool = False, jobs: int = 4) -> dict:
    """Build every variant in ``jobs`` worker processes (scheduling is Python, compiling is
    hipcc; both run in parallel across variants).  The slowest variants start first."""
    from concurrent.futures import ProcessPoolExecutor
    order = sorted(VARIANTS, key=lambda n: ("adj" not in n, n))
    with ProcessPoolExecutor(max_workers=max(1, jobs)) as ex:
        futs = {n: ex.submit(build, n, force) for n in order}
        return {n: f.result() for n, f in futs.items()}


def library(name: str) -> str:
    import os
    from .generator import GEN_DIR
    return os.path.join(GEN_DIR, name, "lib%s.so" % name)


def machine(name: str, local_size):
    from .machine import Machine
    return Machine(library(name), local_size)


def batch(name: str, sizes):
    from .machine import Batch
    return Batch(library(name), sizes)

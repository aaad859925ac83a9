"""Scalar statics that depend on reductions, on several launches and on earlier calls
(paraiso_amd/schemes/monitor.py) against numpy in the program's own precision: the same
operations in the same order, and maxima, are the same bits."""
import ctypes

import numpy as np
import pytest
import torch

from paraiso_amd import variants
from paraiso_amd.machine import load_runtime
from paraiso_amd.schemes.monitor import SIDES

pytestmark = pytest.mark.gpu
# tiles of 32x8: a few, more than a launch folds (1024), more than a call of a run folds (2048)
SIZES = [(40, 23), (700, 500), (1100, 520)]


def field(nx, ny, seed):
    return 0.5 + np.random.default_rng(seed).random((ny, nx))


def relaxed(f):
    a, b, c, d = (np.roll(f, (v[1], v[0]), (0, 1)) for v in SIDES)
    return 0.25 * (a + b + c + d)


class Model:
    def __init__(self, f):
        self.s = {k: 0.0 for k in ("top", "low", "now", "last", "older", "high")}
        self.s.update(weight=1.75, calls=0)
        self.f = f

    def run(self, kernel):
        s, f = self.s, self.f
        if kernel == "normalize":
            s["top"], self.f = f.max(), f / f.max()
            s["low"] = self.f.min()
        elif kernel == "damp":
            s["top"], self.f = f.max(), f * s["weight"] / f.max()
            s["weight"] = 0.5 * s["weight"]
        else:
            self.f = relaxed(f)
            if kernel == "watch":
                s["now"], s["last"], s["older"] = self.f.max(), s["now"], s["last"]
                s["calls"] += 1
            else:
                s["high"] = max(s["high"], self.f.max())


def check(m, model):
    assert np.array_equal(m.get("f"), model.f)
    assert {k: m.get(k) for k in model.s} == model.s


@pytest.mark.parametrize("size", SIZES)
@pytest.mark.parametrize("kernel", ["normalize", "damp"])
def test_two_launches(require_gpu, size, kernel):
    print("monitor %s %s" % (kernel, size), flush=True)
    m, model = variants.machine("monitor_f64", size), Model(field(*size, 3))
    m.set("f", model.f)
    m.set("weight", model.s["weight"])
    for count, graph in ((1, False), (1, False), (3, False), (2, True), (2, True)):
        m.run(kernel, count, graph=graph)
        for _ in range(count):
            model.run(kernel)
        check(m, model)


@pytest.mark.parametrize("size", SIZES[:2])
def test_two_launches_that_allocate_nothing(require_gpu, size):
    print("monitor noalloc %s" % (size,), flush=True)
    rt = load_runtime()
    m, model = variants.machine("monitor_f64", size), Model(field(*size, 4))
    ns, (nx, ny) = len(m.statics), size
    bufs = [torch.from_numpy(model.f).cuda(), torch.zeros((ny, nx), dtype=torch.float64,
                                                          device="cuda")]
    scal = torch.zeros(ns, dtype=torch.float64, device="cuda")
    ptrs = (ctypes.c_void_p * (2 * ns))()
    ptrs[0], ptrs[1] = (b.data_ptr() for b in bufs)
    parity, err = (ctypes.c_int * ns)(), ctypes.create_string_buffer(512)
    rt.pr_run_noalloc.argtypes = [ctypes.c_void_p, ctypes.POINTER(ctypes.c_int), ctypes.c_int,
                                  ctypes.c_int, ctypes.POINTER(ctypes.c_void_p),
                                  ctypes.POINTER(ctypes.c_int), ctypes.c_void_p, ctypes.c_void_p,
                                  ctypes.c_char_p, ctypes.c_size_t]
    torch.cuda.synchronize()
    rc = rt.pr_run_noalloc(ctypes.cast(m.desc_ptr, ctypes.c_void_p),
                           (ctypes.c_int * 3)(nx, ny, 1), m.kernel_index("normalize"), 2, ptrs,
                           parity, ctypes.c_void_p(scal.data_ptr()), None, err, len(err))
    assert rc == 0, err.value
    torch.cuda.synchronize()
    model.run("normalize")
    model.run("normalize")
    assert np.array_equal(bufs[parity[0]].cpu().numpy(), model.f)
    got = scal.cpu().numpy()
    assert [got[m.static_index(k)] for k in ("top", "low")] == [model.s["top"], model.s["low"]]


@pytest.mark.parametrize("size", SIZES)
@pytest.mark.parametrize("kernel", ["watch", "record"])
def test_runs_of_calls(require_gpu, size, kernel):
    """A run leaves what single calls leave, of this call and of those before it."""
    print("monitor %s %s" % (kernel, size), flush=True)
    m, model = variants.machine("monitor_f64", size), Model(field(*size, 5))
    m.set("f", model.f)
    m.set("weight", model.s["weight"])
    for count, graph in ((1, False), (2, False), (5, False), (3, True), (3, True), (1, False)):
        m.run(kernel, count, graph=graph)
        for _ in range(count):
            model.run(kernel)
        check(m, model)


@pytest.mark.parametrize("count", [1, 40])
def test_batches_whose_tiles_do_not_divide(require_gpu, count):
    """Tiles of ten steps over workgroups of four waves, split over the waves (a few tiles) or
    a wave's each (more than eight a CU)."""
    sizes = [(300, 251), (61, 9), (62, 10), (63, 11), (5, 7)] * count
    sizes += [(1900, 1210)] * (count // 20)
    print("monitor batch of %d" % len(sizes), flush=True)
    b = variants.batch("monitor_f64_batch", sizes)
    models = [Model(field(nx, ny, g)) for g, (nx, ny) in enumerate(sizes)]
    for m, model in zip(b.grids, models):
        m.set("f", model.f)
        m.set("weight", model.s["weight"])
    for kernel in ("watch", "normalize", "damp", "record", "watch", "watch"):
        b.run(kernel)
        for model in models:
            model.run(kernel)
    b.sync()
    for m, model in zip(b.grids, models):
        check(m, model)


@pytest.mark.parametrize("count", [1, 2, 3, 4, 5, 8, 11])
def test_fused_kernels_that_have_fused_kernels(require_gpu, count):
    """``watch`` has a kernel for two calls, and that one another for two of its own."""
    print("monitor fused run of %d" % count, flush=True)
    m, model = variants.machine("monitor_f64_batch", (150, 77)), Model(field(150, 77, 6))
    m.set("f", model.f)
    m.set("weight", model.s["weight"])
    for graph in (False, True, True):
        m.run("watch", count, graph=graph)
        for _ in range(count):
            model.run("watch")
        check(m, model)


def test_batches_of_few_tiles(require_gpu):
    """A tile of ten steps over the eight waves of two workgroups: two each, some none."""
    sizes = [(61, 9), (130, 47), (62, 25), (7, 3)]
    print("monitor batch of %s" % (sizes,), flush=True)
    b = variants.batch("monitor_f64_batch", sizes)
    models = [Model(field(nx, ny, g)) for g, (nx, ny) in enumerate(sizes)]
    for m, model in zip(b.grids, models):
        m.set("f", model.f)
        m.set("weight", model.s["weight"])
    for kernel in ("watch", "normalize", "damp", "record", "watch", "watch"):
        b.run(kernel, 2, graph=kernel == "watch")
        for model in models:
            model.run(kernel)
            model.run(kernel)
    b.sync()
    for m, model in zip(b.grids, models):
        check(m, model)

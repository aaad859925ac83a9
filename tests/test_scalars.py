"""Where the generated code leaves a finish kernel out, nothing reads what it would have
written (paraiso_amd/schemes/monitor.py holds a kernel of every kind)."""
import re

import pytest

from paraiso_amd import variants
from paraiso_amd.generator import _hip_sources


def source(variant):
    mk, _, precise = variants.VARIANTS[variant]
    return _hip_sources(variants.setup_of(variant), mk(), precise)[1]


def body(src, head):
    at = src.index(head)
    return src[at:src.index("\n}\n", at)]


@pytest.mark.parametrize("kernel", ["normalize", "damp"])
def test_a_finish_reads_only_slots_that_are_written(kernel):
    """The second launch's finish reads the first launch's scalars from their slots, which only
    the first launch's finish writes: it runs whatever the number of partials."""
    src = source("monitor_f64")
    fin = body(src, "Monitor_%s_l1_fin(" % kernel)
    slots = [int(x) for x in re.findall(r"\(a\.scal \+ (\d+)\);", fin)]
    statics = 8 * len(variants.VARIANTS["monitor_f64"][0]().setup.static_values)
    assert any(x >= statics for x in slots)              # it does read a slot
    launch = body(src, "static int launch_Monitor_%s_l0(" % kernel)
    line = next(ln for ln in launch.splitlines() if "_l0_fin" in ln)
    assert "if" not in line, line


def test_the_hydro_step_needs_no_finish_between_its_launches():
    launch = body(source("hydro_f64"), "static int launch_Hydro_proceed_l0(")
    assert "if (!c->fold || !c->fold->n) hipLaunchKernelGGL(Hydro_proceed_l0_fin" in launch


@pytest.mark.parametrize("kernel", ["watch", "record"])
def test_a_store_of_an_earlier_reduction_is_not_left_to_the_end(kernel):
    """``last`` and ``older`` hold reductions of earlier calls, ``high`` of them all: the last
    call of a run cannot store them from its own reduction alone."""
    fin = body(source("monitor_f64"), "Monitor_%s_l0_fin(" % kernel)
    assert "a.repeat" not in fin


def test_life_stores_its_scalars_at_the_end_of_a_run():
    assert "it < a.repeat" in body(source("life_i32"), "Life_proceed_l0_fin(")

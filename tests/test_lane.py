"""The register-streaming plan (generator/hip/lane.py) on the CPU: every value of the plan,
read where the plan says, is the lowered kernel's, and nothing is read before it is computed,
after it is dropped, or from a lane that does not hold it."""
from fractions import Fraction

import numpy as np
import pytest

from paraiso_amd import annotation as A, variants
from paraiso_amd.generator.hip.ir import lower_kernel
from paraiso_amd.generator.hip.lane import WAVE, plan_lane
from paraiso_amd.generator.native import Language, Setup
from paraiso_amd.generator.plan import translate
from paraiso_amd.om.arith import Op
from paraiso_amd.om.dyn import CType, Realm
from paraiso_amd.schemes.hydro import hydro_om
from paraiso_amd.schemes.life import life_om
from test_merge_selects import BIN


def apply(n_op, cast, a, ctype):
    r = (BIN[n_op](*a) if n_op in BIN else np.where(*a) if n_op is Op.Select else
         np.sqrt(a[0]) if n_op is Op.Sqrt else np.abs(a[0]) if n_op is Op.Abs else
         np.logical_not(a[0]) if n_op is Op.Not else -a[0] if n_op is Op.Neg else
         np.asarray(a[0]).astype(cast.np_dtype) if n_op is Op.Cast else None)
    return r if ctype is CType.Bool else np.asarray(r).astype(ctype.np_dtype)


def lowered(om, kernel, ndim):
    om = translate(Setup((20,) * ndim, Language.HIP, boundary=(A.Condition.Cyclic,) * ndim), om).om
    ki = [k.name for k in om.kernels].index(kernel)
    return om, lower_kernel(om, ki, (True,) * ndim)


CASES = [("hydro", lambda: hydro_om(CType.Double, Fraction(7, 5), "fixed"), "proceed", 2, 1),
         ("life", life_om, "proceed", 2, 1),
         ("wave", variants._wave_adj(3, CType.Double), "proceed_x2", 3, 4),
         ("wave", variants._wave_adj(3, CType.Double), "proceed_adjoint_x2", 3, 5)]


@pytest.mark.parametrize("name,mk,kernel,ndim,rows", CASES)
@pytest.mark.parametrize("prefetch", [1, 2])
def test_plan(name, mk, kernel, ndim, rows, prefetch):
    om, k = lowered(mk(), kernel, ndim)
    shape = (14, 12, 10)[:ndim]
    axes = tuple(reversed(range(ndim)))             # OM axis 0 is the array's last
    rng = np.random.default_rng(3)
    stat = {}
    for i, s in enumerate(om.setup.static_values):
        x = 1 + np.abs(rng.standard_normal(shape)) if s.dyn.realm is Realm.Array else 0.05
        if s.dyn.ctype is CType.Int:
            x = rng.integers(0, 2, shape) if s.dyn.realm is Realm.Array else 2
        stat[i] = np.asarray(x).astype(s.dyn.ctype.np_dtype)
    at = lambda a, off: np.roll(a, [-o for o in off], axes)      # value read at an offset
    val = {}
    for n in k.nodes:
        a = [val[x] for x in n.args]
        val[n.id] = (stat[n.payload] if n.op == "load" else
                     np.asarray(n.payload) if n.op == "imm" else
                     np.broadcast_to(a[0], shape) if n.op == "bcast" else
                     at(a[0], [-v for v in n.payload]) if n.op == "shift" else
                     a[0].sum() if n.op == "reduce" else
                     apply(n.payload[0], n.payload[1], a, n.ctype))
    targets = sorted(set(v for _, v in k.stores if k.nodes[v].realm is Realm.Array)
                     | set(n.args[0] for n in k.nodes if n.op == "reduce"))
    p = plan_lane(k, targets, rows, prefetch)
    assert p is not None and p.width >= 8
    got, by_id = {}, {v.id: v for v in p.values}

    def uniform(u):
        return val[int(u[1:])]
    for v in p.values:
        if v.op == "load":
            got[v.id] = stat[v.payload]
        else:
            args = [uniform(b) if o is None else at(got[b], o) for b, o in v.args]
            got[v.id] = apply(v.payload[0], v.payload[1], args, v.ctype)

    def check(b, place, lead, off, r, first, lo, hi):
        w = by_id[b]
        delay = w.lead - lead - off[ndim - 1]
        assert (prefetch if w.op == "load" else 0) <= delay <= w.depth
        assert w.first <= first - delay
        assert r + (off[1] if ndim == 3 else 0) in w.rows
        dx = place + off[0] - w.place
        assert w.lanes[0] <= lo + dx and hi + dx <= w.lanes[1]
        assert 0 <= w.lanes[0] <= w.lanes[1] < WAVE
    for v in p.values:
        for b, o in v.args:
            if o is not None:
                for r in v.rows:
                    check(b, v.place, v.lead, o, r, v.first, *v.lanes)
    for t, (b, o) in p.targets.items():
        assert np.array_equal(at(got[b], o), val[t]), t
        for r in range(rows if ndim == 3 else 1):
            check(b, 0, 0, o, r, 0, *p.lanes)

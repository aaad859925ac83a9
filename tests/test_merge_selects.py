"""Selecting before computing (ir.merge_selects) picks the same bits as selecting after.

The lowered kernel is evaluated with numpy before and after the rewrite, on values with
infinities, NaNs, signed zeros and sign changes, so that every branch of every chain is taken.
"""
from fractions import Fraction

import numpy as np
import pytest

from paraiso_amd import annotation as A
from paraiso_amd.generator.hip.ir import lower_kernel
from paraiso_amd.generator.native import Language, Setup
from paraiso_amd.generator.plan import translate
from paraiso_amd.om.arith import Op
from paraiso_amd.om.dyn import CType, Realm
from paraiso_amd.schemes.hydro import hydro_om

BIN = {Op.Add: np.add, Op.Sub: np.subtract, Op.Mul: np.multiply, Op.Div: np.divide,
       Op.LT: np.less, Op.LE: np.less_equal, Op.GT: np.greater, Op.GE: np.greater_equal,
       Op.EQ: np.equal, Op.NE: np.not_equal, Op.And: np.logical_and, Op.Or: np.logical_or,
       Op.Max: lambda a, b: np.where(a < b, b, a), Op.Min: lambda a, b: np.where(b < a, b, a)}


def evaluate(k, statics):
    val = []
    with np.errstate(all="ignore"):
        for n in k.nodes:
            a = [val[x] for x in n.args]
            if n.op == "load":
                r = statics[n.payload]
            elif n.op == "imm":
                r = n.payload
            elif n.op == "shift":
                r = np.roll(a[0], n.payload, tuple(range(k.ndim)))
            elif n.op == "bcast":
                r = np.broadcast_to(a[0], (12, 10))
            elif n.op == "reduce":
                r = a[0].min()
            else:
                op, cast = n.payload
                r = (BIN[op](*a) if op in BIN else np.where(*a) if op is Op.Select else
                     np.sqrt(a[0]) if op is Op.Sqrt else np.abs(a[0]) if op is Op.Abs else
                     np.logical_not(a[0]) if op is Op.Not else -a[0] if op is Op.Neg else None)
            if n.ctype is not CType.Bool and n.ctype is not CType.Int:
                r = np.asarray(r, dtype=n.ctype.np_dtype)
            val.append(r)
    return [val[v] for _, v in k.stores]


@pytest.mark.parametrize("real", [CType.Float, CType.Double])
@pytest.mark.parametrize("special", [False, True])
def test_hydro_step_keeps_its_bits(real, special):
    om = translate(Setup((12, 10), Language.HIP, boundary=(A.Condition.Cyclic,) * 2),
                   hydro_om(real, Fraction(7, 5))).om
    ki = [k.name for k in om.kernels].index("proceed")
    before = lower_kernel(om, ki, (True, True), merge=False)
    after = lower_kernel(om, ki, (True, True))
    count = lambda k: sum(n.op == "arith" for n in k.nodes)
    assert count(after) < 0.92 * count(before)
    rng = np.random.default_rng(5)
    statics = {}
    for i, s in enumerate(om.setup.static_values):
        if s.dyn.realm is Realm.Array:
            x = rng.standard_normal((12, 10)) * (3 if "velocity" in s.name else 0.3)
            x = x if "velocity" in s.name else 1 + np.abs(x)
            if special:
                x[2, 3], x[5, 5], x[7, 1], x[9, 9] = np.inf, np.nan, -0.0, -2.0
            statics[i] = x.astype(real.np_dtype)
        else:
            statics[i] = real.np_dtype(0.1) if s.dyn.ctype is real else 3
    assert [s for s, _ in before.stores] == [s for s, _ in after.stores]
    for a, b in zip(evaluate(before, statics), evaluate(after, statics)):
        assert np.array_equal(a, b, equal_nan=True)

"""A relaxation whose scalar statics watch it: every way in which a kernel's stored scalars
depend on its reductions, on its own launches and on what the calls before it stored.

* ``normalize``, ``damp``: the stored array needs a reduction of the loaded one, and the
  scalar statics need both that reduction and one of the result (``normalize``) or a scalar
  that the kernel also stores (``damp``),
* ``watch``: the extreme of this call, of the call before and of the one before that,
* ``record``: the extreme over all calls.

Only maxima and minima are reduced, so that the results are the same bits in any order.
"""
from __future__ import annotations

from ..om import builder as B
from ..om.arith import ReduceOp
from ..om.dyn import CType, Realm

SIDES = ((1, 0), (-1, 0), (0, 1), (0, -1))


def monitor_om(real: CType = CType.Double, name: str = "Monitor"):
    f = B.static("f", Realm.Array, real)
    scalars = [B.static(n, Realm.Scalar, real)
               for n in ("top", "low", "weight", "now", "last", "older", "high")]
    calls = B.static("calls", Realm.Scalar, CType.Int)
    top, low, weight, now, last, older, high = scalars

    def relaxed():
        f0 = B.bind(B.load(f))
        side = [B.bind(B.shift(v, f0)) for v in SIDES]
        return B.bind(0.25 * (side[0] + side[1] + side[2] + side[3]))

    def normalize():
        f0 = B.bind(B.load(f))
        t = B.bind(B.reduce(ReduceOp.Max, f0))
        f1 = B.bind(f0 / B.broadcast(t))
        B.store(f, f1)
        B.store(top, t)
        B.store(low, B.reduce(ReduceOp.Min, f1))

    def damp():
        f0 = B.bind(B.load(f))
        w = B.bind(B.load(weight))
        t = B.bind(B.reduce(ReduceOp.Max, f0))
        B.store(f, f0 * B.broadcast(w) / B.broadcast(t))
        B.store(top, t)
        B.store(weight, 0.5 * w)

    def watch():
        f1 = relaxed()
        n, p, c = (B.bind(B.load(x)) for x in (now, last, calls))
        B.store(f, f1)
        B.store(now, B.reduce(ReduceOp.Max, f1))
        B.store(last, n)
        B.store(older, p)
        B.store(calls, c + 1)

    def record():
        f1 = relaxed()
        h = B.bind(B.load(high))
        B.store(f, f1)
        B.store(high, B.max_(h, B.reduce(ReduceOp.Max, f1)))

    return B.make_om(name, [], [f] + scalars + [calls],
                     [("normalize", normalize), ("damp", damp), ("watch", watch),
                      ("record", record)], ndim=2)

"""A program of the expressions that a fast FP32 streaming build evaluates in another form
(``generator/hip/lane.py``): the minmod limiter, quotients with a common divisor, a quotient
by one of two values that are divided by anyway, and the maximum of a number and a value."""
from __future__ import annotations

from ..om import builder as B
from ..om.dyn import CType, Realm

OUT = ("limited", "shifted", "ratio_a", "ratio_b", "ratio_d", "picked", "floored")


def rewrites_om(name: str = "Rewrites"):
    by = {n: B.static(n, Realm.Array, CType.Float) for n in ("a", "b", "c", "d") + OUT}

    def minmod(x, y):
        return B.select((x * y).le(0), 0, B.select(B.abs_(x).lt(B.abs_(y)), x, y))

    def apply():
        a, b, c, d = (B.bind(B.load(by[n])) for n in ("a", "b", "c", "d"))
        right = B.bind(B.shift((-1, 0), b))
        B.store(by["limited"], minmod(a, b))
        B.store(by["shifted"], minmod(a, right))
        B.store(by["ratio_a"], a / c)
        B.store(by["ratio_b"], b / c)
        B.store(by["ratio_d"], b / d)
        B.store(by["picked"], a / B.bind(B.select(a.lt(b), c, d)))
        B.store(by["floored"], B.max_(0.5, a))

    return B.make_om(name, [], list(by.values()), [("apply", apply)], ndim=2)

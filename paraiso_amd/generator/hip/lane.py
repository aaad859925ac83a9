"""Register streaming: the launch form in which a wave keeps its whole stencil in registers.

A wave64 owns a strip of the grid: its lanes are neighbouring cells along x, in three
dimensions each lane holds a few rows along y, and the wave streams along the last axis, one
row (2-D) or plane (3-D) per step.  A value read at another x comes from the neighbouring
lane by a DPP move, at another y from another register of the lane, and at another position
of the streaming axis from the register that kept it from an earlier step.  Nothing goes
through LDS, there is no barrier, the addresses are scalar, and every value of the kernel is
computed once per cell (the outermost lanes, and rows, of a strip excepted).

``plan_lane`` turns a launch into that form:

1. values are numbered up to translation: ``op(shift(a, v), shift(b, v))`` and ``shift(op(a,
   b), v)`` are the same value read at two places, so what the program derives again from a
   shifted state (a sound speed, an energy) is derived once,
2. each value gets a *placement*: the offset, from the cell being stored, of the cell it is
   computed for.  Along x the placement decides which reads need a lane move; along the
   streaming axis it decides how many steps a value is kept (its readers run behind it),
3. the lanes whose results are complete follow from the moves; the others are the overlap
   between neighbouring strips.
"""
from __future__ import annotations

from dataclasses import dataclass, field
from typing import Dict, List, Optional, Set, Tuple

from ...om.dyn import CType, Realm
from .ir import LKernel

WAVE = 64


@dataclass
class LaneValue:
    id: int
    op: str                                   # load index arith
    args: List[Tuple[object, Tuple[int, ...]]]   # (value id, offset) or (uniform name, None)
    ctype: CType
    payload: object
    node: int                                 # a node of the lowered kernel it stands for
    place: int = 0                            # x placement
    lead: int = 0                             # streaming-axis placement
    first: int = 0                            # first step that computes it (0: first store)
    depth: int = 0                            # steps it is kept after its own
    rows: Tuple[int, ...] = (0,)              # y rows a lane computes (3-D)
    lanes: Tuple[int, int] = (0, WAVE - 1)


@dataclass
class LanePlan:
    values: List[LaneValue]
    uniform: List[int]                        # array values that hold one number (node ids)
    targets: Dict[int, Tuple[int, Tuple[int, ...]]]   # target node -> (value, offset)
    uniform_targets: Set[int]
    lanes: Tuple[int, int]                    # lanes that store
    first: int                                # first step (<= 0)
    ndim: int
    rows: int
    prefetch: int
    reach: int

    @property
    def width(self) -> int:
        return self.lanes[1] - self.lanes[0] + 1


def plan_lane(k: LKernel, targets: List[int], rows: int = 1, prefetch: int = 1
              ) -> Optional[LanePlan]:
    """The register-streaming plan of the values ``targets`` of one launch, or None when the
    launch has no array value to read (nothing to stream)."""
    nd = k.ndim
    if nd not in (2, 3):
        return None
    zero = (0,) * nd
    nodes = k.nodes
    cone, stack = set(), list(targets)
    while stack:
        x = stack.pop()
        if x in cone:
            continue
        cone.add(x)
        n = nodes[x]
        if n.op in ("arith", "shift") and n.realm is Realm.Array:
            stack.extend(n.args)
    values: List[LaneValue] = []
    memo: Dict[tuple, int] = {}
    where: Dict[int, Tuple[object, Optional[Tuple[int, ...]]]] = {}
    uniform: List[int] = []

    def add(op, args, ct, payload, node):
        key = (op, tuple(args), ct, payload if op != "arith" else (payload[0], payload[1]))
        if key not in memo:
            memo[key] = len(values)
            values.append(LaneValue(len(values), op, list(args), ct, payload, node))
        return memo[key]

    for v in sorted(cone):
        n = nodes[v]
        if n.realm is not Realm.Array or n.op in ("imm", "bcast", "size"):
            uniform.append(v)
            where[v] = ("n%d" % v, None)
        elif n.op in ("load", "index"):
            where[v] = (add(n.op, (), n.ctype, n.payload, v), zero)
        elif n.op == "shift":
            b, o = where[n.args[0]]
            where[v] = (b, None if o is None else tuple(x - y for x, y in zip(o, n.payload)))
            if o is None:
                where[v] = (b, None)
        elif n.op == "arith":
            ps = [where[a] for a in n.args]
            origin = next((o for _, o in ps if o is not None), None)
            if origin is None:
                uniform.append(v)
                where[v] = ("n%d" % v, None)
                continue
            args = tuple((b, None if o is None else tuple(x - y for x, y in zip(o, origin)))
                         for b, o in ps)
            where[v] = (add("arith", args, n.ctype, n.payload, v), origin)
        else:
            raise NotImplementedError(n.op)
    tgt = {t: where[t] for t in targets if where[t][1] is not None}
    uniform_targets = set(t for t in targets if where[t][1] is None)
    if not any(v.op == "load" for v in values):
        return None
    ma = nd - 1
    users: Dict[int, List[Tuple[Optional[int], Tuple[int, ...]]]] = {v.id: [] for v in values}
    for v in values:
        for b, o in v.args:
            if o is not None:
                users[b].append((v.id, o))
    for b, o in tgt.values():
        users[b].append((None, o))
    live = set()
    stack = [b for b, _ in tgt.values()]
    while stack:
        x = stack.pop()
        if x not in live:
            live.add(x)
            stack.extend(b for b, o in values[x].args if o is not None)

    def want(u, o, axis):
        """Offset at which a reader wants a value, along the axis."""
        if u is None:
            return o[axis]
        w = values[u]
        return o[axis] + (w.place if axis == 0 else w.lead)

    order = [v for v in values if v.id in live]
    keep = lambda v: prefetch if v.op == "load" else 0      # loads are issued ahead
    # ---- streaming axis: readers first, each value as late as its readers allow, then
    # earlier where that keeps fewer registers (it stands in for its own inputs)
    for v in reversed(order):
        v.lead = max(want(u, o, ma) for u, o in users[v.id] if u is None or u in live) + keep(v)

    def depth(v):
        return max(v.lead - want(u, o, ma) for u, o in users[v.id] if u is None or u in live)

    def weight(v):
        return v.ctype.size / 4.0 if v.ctype is not CType.Bool else 1.0

    def kept(v):
        ins = set(b for b, o in v.args if o is not None)
        return sum(weight(values[b]) * depth(values[b]) for b in ins) + weight(v) * depth(v)
    for _ in range(12):
        moved = False
        for v in order:
            if v.op == "load":
                continue
            best, base = kept(v), v.lead
            choice = base
            least = max(want(u, o, ma) for u, o in users[v.id] if u is None or u in live)
            most = min([values[b].lead - keep(values[b]) - o[ma] for b, o in v.args
                        if o is not None] + [base if v.op == "index" else 1 << 20])
            for lead in range(least, most + 1):
                v.lead = lead
                c = kept(v)
                if c < best - 1e-9:
                    best, choice = c, lead
            v.lead = choice
            moved |= choice != base
        for v in order:
            if v.op == "load":
                v.lead = max(want(u, o, ma) for u, o in users[v.id]
                             if u is None or u in live) + keep(v)
        if not moved:
            break
    # ---- x: each value where most of its readers want it, then moved while that saves moves
    for v in reversed(order):
        xs = [want(u, o, 0) for u, o in users[v.id] if u is None or u in live]
        v.place = max(sorted(set(xs)), key=xs.count)

    def moves(b):
        w = values[b]
        return sum(abs(d) for d in set(
            want(u, o, 0) - w.place for u, o in users[b] if u is None or u in live)) * weight(w)

    def local(v):
        return moves(v.id) + sum(moves(b) for b in set(b for b, o in v.args if o is not None))
    for _ in range(12):
        moved = False
        for v in order:
            base = v.place
            best, choice = local(v), base
            for p in range(base - 2, base + 3):
                v.place = p
                c = local(v)
                if c < best - 1e-9:
                    best, choice = c, p
            v.place = choice
            moved |= choice != base
        if not moved:
            break
    # ---- steps, kept registers, rows and lanes
    for v in order:
        v.depth = depth(v)
    rows_of: Dict[int, Set[int]] = {v.id: set() for v in order}
    firsts: Dict[int, int] = {}
    for b, o in tgt.values():
        rows_of[b] |= set(r + (o[1] if nd == 3 else 0) for r in range(rows))
    for v in reversed(order):
        f = []
        for u, o in users[v.id]:
            if u is None:
                f.append(o[ma] - v.lead)
            elif u in live:
                f.append(values[u].first + values[u].lead + o[ma] - v.lead)
                rows_of[v.id] |= set(r + (o[1] if nd == 3 else 0) for r in rows_of[u])
        v.first = min(f)
        v.rows = tuple(sorted(rows_of[v.id]))
    for v in order:
        lo, hi = 0, WAVE - 1
        for b, o in v.args:
            if o is None:
                continue
            d = o[0] + v.place - values[b].place
            lo = max(lo, values[b].lanes[0] - d)
            hi = min(hi, values[b].lanes[1] - d)
        v.lanes = (max(lo, 0), min(hi, WAVE - 1))
    lo, hi = 0, WAVE - 1
    for b, o in tgt.values():
        d = o[0] - values[b].place
        lo, hi = max(lo, values[b].lanes[0] - d), min(hi, values[b].lanes[1] - d)
    if hi - lo < 8:
        return None
    reach = 1
    for v in order:
        reach = max([reach, abs(v.place), abs(v.lead), abs(v.lead + v.first)]
                    + [abs(r) for r in v.rows])
    return LanePlan(order, uniform, tgt, uniform_targets, (lo, hi),
                    min(v.first for v in order), nd, rows, prefetch, reach)


def registers(p: LanePlan) -> int:
    """32-bit registers the values kept from step to step take, per lane."""
    return sum(v.depth * len(v.rows) * max(1, v.ctype.size // 4) for v in p.values)

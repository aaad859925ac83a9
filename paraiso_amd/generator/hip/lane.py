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

from ...om.arith import Op
from ...om.dyn import CType, Realm
from .ir import LKernel

WAVE = 64


@dataclass
class LaneValue:
    id: int
    op: str                                   # load index arith
    args: List[Tuple[object, Tuple[int, ...]]]   # (value id, offset) or (uniform name, None)
    ctype: CType
    payload: object                           # static, axis, or (operator, cast)
    consts: List[object]                      # per argument: its exact constant value, or None
    types: List[CType]                        # per argument
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

    @property
    def runup(self) -> float:
        """What the steps before the first store cost, in steps."""
        size = lambda v: len(v.rows) if v.op == "arith" else 0
        return (sum(size(v) * max(0, -v.first) for v in self.values)
                / max(1, sum(size(v) for v in self.values)))


MINMOD = "minmod"             # of fast FP32 plans: see om_minmod


def plan_lane(k: LKernel, targets: List[int], rows: int = 1, prefetch: int = 1,
              fast: bool = False) -> Optional[LanePlan]:
    """The register-streaming plan of the values ``targets`` of one launch, or None when the
    launch has no array value to read (nothing to stream).

    ``fast`` (fast FP32 builds): a division is a product with a reciprocal of its own, which
    other divisions share; the reciprocal of a Select between two values whose reciprocals are
    there anyway is the Select of those (a transcendental instruction takes four slots, a
    select one); and ``a * b <= 0 ? 0 : (|a| < |b| ? a : b)`` is one operation."""
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

    def add(op, args, ct, payload, consts=(), types=()):
        key = (op, tuple(args), ct, payload)
        if key not in memo:
            memo[key] = len(values)
            values.append(LaneValue(len(values), op, list(args), ct, payload, list(consts),
                                    list(types)))
        return memo[key]

    def operation(op, cast, ps, ct, consts, types):
        """(value, offset) of an operation on (value, offset) arguments, one not uniform."""
        origin = next(o for _, o in ps if o is not None)
        args = tuple((b, None if o is None else tuple(x - y for x, y in zip(o, origin)))
                     for b, o in ps)
        return add("arith", args, ct, (op, cast), consts, types), origin

    def reciprocal(p):
        b, o = p
        v = values[b]
        if v.op == "arith" and v.payload[0] is Op.Select and v.args[0][1] is not None:
            c, x, y = v.args
            there = [("arith", ((z[0], zero),), CType.Float, (Op.Inv, None)) for z in (x, y)]
            if all(z[1] is not None and t in memo for z, t in zip((x, y), there)):
                ix, iy = ((memo[t], z[1]) for t, z in zip(there, (x, y)))
                w, ow = operation(Op.Select, None, [c, ix, iy], CType.Float, [None] * 3,
                                  [CType.Bool, CType.Float, CType.Float])
                return w, tuple(i + j for i, j in zip(o, ow))
        return add("arith", ((b, zero),), CType.Float, (Op.Inv, None), [None], [CType.Float]), o

    def minmod(v):
        """(a, b) where value v is a * b <= 0 ? 0 : (|a| < |b| ? a : b), else None."""
        def is_op(p, op):
            return (p[1] == zero and values[p[0]].op == "arith"
                    and values[p[0]].payload[0] is op)
        if v.op != "arith" or v.payload[0] is not Op.Select or v.ctype is not CType.Float:
            return None
        cond, nil, inner = v.args
        if v.consts[1] != 0 or not is_op(cond, Op.LE) or not is_op(inner, Op.Select):
            return None
        le, sel = values[cond[0]], values[inner[0]]
        if le.consts[1] != 0 or not is_op(le.args[0], Op.Mul) or not is_op(sel.args[0], Op.LT):
            return None
        a, b = sel.args[1:]
        lt = values[sel.args[0][0]]
        if set(values[le.args[0][0]].args) != {a, b} or a[1] is None or b[1] is None:
            return None
        for p, x in zip(lt.args, (a, b)):
            if p[1] is None or values[p[0]].op != "arith" or values[p[0]].payload[0] is not Op.Abs:
                return None
            y, oy = values[p[0]].args[0]
            if oy is None or (y, tuple(i + j for i, j in zip(oy, p[1]))) != x:
                return None
        return [a, b]

    for v in sorted(cone):
        n = nodes[v]
        if n.realm is not Realm.Array or n.op in ("imm", "bcast", "size"):
            uniform.append(v)
            where[v] = ("n%d" % v, None)
        elif n.op in ("load", "index"):
            where[v] = (add(n.op, (), n.ctype, n.payload), zero)
        elif n.op == "shift":
            b, o = where[n.args[0]]
            where[v] = (b, None if o is None else tuple(x - y for x, y in zip(o, n.payload)))
        elif n.op == "arith":
            ps = [where[a] for a in n.args]
            if all(o is None for _, o in ps):
                uniform.append(v)
                where[v] = ("n%d" % v, None)
                continue
            op, cast = n.payload
            consts = [k.exact.get(a) for a in n.args]
            types = [nodes[a].ctype for a in n.args]
            if (fast and op is Op.Div and n.ctype is CType.Float and consts[1] is None
                    and ps[1][1] is not None):
                ps = [ps[0], reciprocal(ps[1])]
                op, consts = Op.Mul, [consts[0], None]
            where[v] = operation(op, cast, ps, n.ctype, consts, types)
            m = minmod(values[where[v][0]]) if fast else None
            if m is not None:
                w, o = operation(MINMOD, None, m, CType.Float, [None] * 2, [CType.Float] * 2)
                where[v] = (w, tuple(i + j for i, j in zip(o, where[v][1])))
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


def _n(x: int) -> str:
    return "m%d" % -x if x < 0 else "%d" % x


def fused_products(p: LanePlan, product) -> Dict[int, int]:
    """The multiply-adds of a fast FP32 build: addition or subtraction -> the argument that is
    a product it takes in.  Fixed here rather than left to the compiler, which would choose
    anew in every copy of a step (the run-up, the unrolled loop): a cell's bits must not
    depend on which copy computed it, that is on how the grid was cut into chunks.  A product
    is taken in by all its readers or by none.  ``product(value)``: it may be fused."""
    by_id = {v.id: v for v in p.values}
    users: Dict[int, List[LaneValue]] = {v.id: [] for v in p.values}
    for v in p.values:
        for b, o in v.args:
            if o is not None:
                users[b].append(v)
    targets = set(b for b, _ in p.targets.values())
    out: Dict[int, int] = {}
    for v in p.values:
        if not product(v) or v.id in targets or v.depth or not users[v.id]:
            continue
        spots = []
        for u in users[v.id]:
            i = [j for j, (b, o) in enumerate(u.args) if b == v.id and o is not None]
            if (u.op != "arith" or u.payload[0] not in (Op.Add, Op.Sub) or u.id in out
                    or u.ctype is not CType.Float or len(i) != 1 or any(u.args[i[0]][1])
                    or u.lead != v.lead or u.place != v.place):
                break
            spots.append((u.id, i[0]))
        else:
            out.update(spots)
    return out


class LaneEmitter:
    """The device code of one launch in register-streaming form (see the module's docstring).

    ``load_ptr(static)`` is a static's pointer; ``arith(value, args)`` the C expression of an
    operation; ``stores`` and ``reduces`` list (C pointer, C type, target) and (accumulator,
    operator, C type, initial value, target)."""

    def __init__(self, plan: LanePlan, load_ptr, arith, stores, reduces, fused=None):
        """``fused``: as ``fused_products`` gives it; ``arith`` then gets, in the place of that
        argument, the pair of names it multiplies."""
        self.p = plan
        self.fused = fused or {}
        self.inside = set(self._arg(u, i) for u, i in self.fused.items())
        self.by_id = {v.id: v for v in plan.values}
        self.load_ptr, self.arith = load_ptr, arith
        self.stores, self.reduces = stores, reduces
        self.ma = plan.ndim - 1
        self.lines: List[str] = []

    def _arg(self, u: int, i: int) -> int:
        return next(v for v in self.p.values if v.id == u).args[i][0]

    # ------------------------------------------------------------ names
    def name(self, v: LaneValue, row: int, delay: int) -> str:
        r = "_r%s" % _n(row) if self.p.ndim == 3 else ""
        return "v%d%s" % (v.id, r) if delay == 0 else "h%d%s_%d" % (v.id, r, delay)

    def read(self, b: int, off, place: int, lead: int, row: int, moved: Dict, w) -> str:
        """Value ``b`` at ``off`` from a reader placed at (place, lead), as a C name; lane moves
        are emitted once per step."""
        v = self.by_id[b]
        delay = v.lead - lead - off[self.ma]
        dx = place + off[0] - v.place
        r = row + (off[1] if self.p.ndim == 3 else 0)
        nm = self.name(v, r, delay)
        if dx == 0:
            return nm
        key = (b, r, delay, dx)
        if key not in moved:
            moved[key] = "x%s_%s" % (nm, _n(dx))
            w("const %s %s = om_lane<%d>(%s);" % (v.ctype.c_name, moved[key], dx, nm))
        return moved[key]

    # ------------------------------------------------------------ parts
    def setup(self, width: int) -> List[str]:
        """Per-wave coordinates: the lane's column, the rows' offsets and the kept registers."""
        p, out = self.p, []
        w = out.append
        lo, hi = p.lanes[0], p.lanes[0] + width - 1
        w("const int x = X0 + lane - %d;" % lo)
        w("const bool ok = lane >= %d && lane <= %d && x < a.n0;" % (lo, hi))
        for place in sorted(set(v.place for v in p.values if v.op == "load" or
                                (v.op == "index" and v.payload == 0))):
            w("const int x_%s = om_wrap(x + (%d), a.n0, a.wide);" % (_n(place), place))
        if p.ndim == 3:
            for r in sorted(set(r for v in p.values for r in v.rows)):
                w("const int y_%s = om_wrap(Y0 + (%d), a.n1, a.wide);" % (_n(r), r))
        for v in p.values:
            for r in v.rows:
                if v.depth:
                    w("%s %s;" % (v.ctype.c_name, ", ".join(
                        "%s = (%s)0" % (self.name(v, r, d), v.ctype.c_name)
                        for d in range(1, v.depth + 1))))
        return out

    def step(self, s: str, at: Optional[int], when: str = "") -> List[str]:
        """One step; ``at`` is its number in the run-up before the first store, or None;
        ``when``: a condition on its stores and reductions."""
        p, out = self.p, []
        w = out.append
        on = lambda v: at is None or v.first <= at
        last = "a.n%d" % self.ma
        for lead in sorted(set(v.lead for v in p.values if on(v) and
                               (v.op == "load" or (v.op == "index" and v.payload == self.ma)))):
            w("const int m_%s = om_wrap(S0 + (%s) + (%d), %s, a.wide);" % (_n(lead), s, lead, last))
        moved: Dict = {}
        for v in p.values:
            if not on(v) or v.id in self.inside:
                continue
            tn = v.ctype.c_name
            for r in v.rows:
                nm = self.name(v, r, 0)
                if v.op == "load":
                    row = ("(size_t)m_%s * a.n0" % _n(v.lead) if p.ndim == 2 else
                           "((size_t)m_%s * a.n1 + y_%s) * a.n0" % (_n(v.lead), _n(r)))
                    w("const %s %s = om_at(%s + %s, x_%s);" % (tn, nm, self.load_ptr(v.payload), row,
                                                              _n(v.place)))
                elif v.op == "index":
                    src = ("x_%s" % _n(v.place) if v.payload == 0 else
                           "m_%s" % _n(v.lead) if v.payload == self.ma else "y_%s" % _n(r))
                    w("const %s %s = (%s)%s;" % (tn, nm, tn, src))
                else:
                    def names(u):
                        return [b if o is None else self.read(b, o, u.place, u.lead, r, moved, w)
                                for b, o in u.args]
                    i = self.fused.get(v.id)
                    args = [b if o is None else None if j == i else
                            self.read(b, o, v.place, v.lead, r, moved, w)
                            for j, (b, o) in enumerate(v.args)]
                    if i is not None:
                        args[i] = (self.by_id[v.args[i][0]], names(self.by_id[v.args[i][0]]))
                    w("const %s %s = %s;" % (tn, nm, self.arith(v, args)))
        if at is None:
            rows = range(p.rows) if p.ndim == 3 else [0]
            for r in rows:
                pre = []
                def target(t):
                    if t in p.uniform_targets:
                        return "n%d" % t
                    b, o = p.targets[t]
                    return self.read(b, o, 0, 0, r, moved, pre.append)
                vals = [target(t) for _, _, t in self.stores]
                reds = [target(t) for _, _, _, _, t in self.reduces]
                out.extend(pre)
                cond = [when] * bool(when) + ["Y0 + %d < a.n1" % r] * (p.ndim == 3)
                if cond:
                    w("if (%s) {" % " && ".join(cond))
                if self.stores:
                    w("if (ok) {")
                    row = ("(size_t)(S0 + (%s)) * a.n0" % s if p.ndim == 2 else
                           "((size_t)(S0 + (%s)) * a.n1 + (Y0 + %d)) * a.n0" % (s, r))
                    for (ptr, tn, _), val in zip(self.stores, vals):
                        w("  om_put(%s + %s, x, (%s)%s);" % (ptr, row, tn, val))
                    w("}")
                for (acc, op, tn, init, _), val in zip(self.reduces, reds):
                    w("%s = %s(%s, ok ? (%s)%s : (%s)%s);" % (acc, op, acc, tn, val, tn, init))
                if cond:
                    w("}")
        for v in p.values:
            if on(v):
                for r in v.rows:
                    for d in range(v.depth, 0, -1):
                        w("%s = %s;" % (self.name(v, r, d), self.name(v, r, d - 1)))
        return out

    def body(self, width: int, peel: bool = True) -> List[str]:
        """The steps of a wave: the run-up, each step with only the values that something reads
        later, then the loop.  Without ``peel`` the loop runs the run-up too (less code)."""
        out = ["    " + ln for ln in self.setup(width)]
        first = 0 if peel else self.p.first
        for s in range(self.p.first, first):
            out.append("    {  // run-up, step %d" % s)
            out += ["      " + ln for ln in self.step("%d" % s, s)]
            out.append("    }")
        out.append("#pragma unroll 1")
        out.append("    for (int s = %d; s < H; ++s) {" % first)
        out += ["      " + ln for ln in self.step("s", None, "" if peel else "s >= 0")]
        out.append("    }")
        return out

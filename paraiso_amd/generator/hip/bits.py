"""Bit planes: the launch form for cellular automata, whose cells hold 0 or 1.

A wave64 owns a square of 64 x 64 cells.  It reads the rows with its lanes along x and turns
them with ballots so that lane r holds row r as 64 bits, in two registers; a cell's neighbour
along x is then a bit shift, along y a lane move (DPP), and one bitwise instruction works on
32 cells of 64 rows.  A value that counts (a sum of neighbours) is a few planes, one per binary
digit, added with carry-save adders; a comparison with a constant is a formula of its planes.

The cells of the program are integers, which may hold anything: a wave that reads another
value than 0 or 1 computes its square by register streaming instead (``lane.py``).

``plan_bits`` gives None for a launch that is not such an automaton: whose values are not all
integers with small known ranges and booleans, or that compares with anything but constants.
"""
from __future__ import annotations

from dataclasses import dataclass
from typing import Dict, List, Optional, Tuple

from ...om.arith import COMPARISONS, Op, ReduceOp
from ...om.dyn import CType
from .ir import LKernel
from .lane import LanePlan, _n

SIDE = 64
MOST = 15                     # largest count a value may reach (four planes)


@dataclass
class BitPlan:
    lane: LanePlan
    top: Dict[int, int]                       # value -> largest number it holds
    const: Dict[str, int]                     # uniform name -> value
    cols: Tuple[int, int]                     # bits, and
    rows: Tuple[int, int]                     # lanes, of a square whose results are complete

    @property
    def width(self) -> int:
        return self.cols[1] - self.cols[0] + 1

    @property
    def height(self) -> int:
        return self.rows[1] - self.rows[0] + 1


def plan_bits(k: LKernel, lane: Optional[LanePlan], stores, reduces) -> Optional[BitPlan]:
    """``stores`` and ``reduces``: the target nodes stored, and (operator, node) reduced."""
    if lane is None or lane.ndim != 2 or lane.uniform_targets:
        return None
    const = {}
    for v in lane.uniform:
        n = k.nodes[v]
        if n.op == "imm" and n.ctype in (CType.Int, CType.Bool):
            const["n%d" % v] = int(n.payload)
    top: Dict[int, int] = {}
    box: Dict[int, Tuple[int, int, int, int]] = {}
    for v in lane.values:
        known = [const.get(b) if o is None else top.get(b) for b, o in v.args]
        if any(x is None or x < 0 for x in known):
            return None
        if v.op == "load":
            if v.ctype is not CType.Int:
                return None
            t = 1
        elif v.op == "index":
            return None
        else:
            op = v.payload[0]
            if op is Op.Add:
                t = sum(known)
            elif op in COMPARISONS:
                if sum(o is None for _, o in v.args) != 1:
                    return None
                t = 1
            elif op in (Op.And, Op.Or, Op.Not):
                if v.ctype is not CType.Bool:
                    return None
                t = 1
            elif op is Op.Select:
                if v.args[0][1] is None:
                    return None
                t = max(known[1:])
            else:
                return None
        if t > MOST:
            return None
        top[v.id] = t
        b = [0, SIDE - 1, 0, SIDE - 1]
        for a, o in v.args:
            if o is not None:
                c = box[a]
                b = [max(b[0], c[0] - o[0]), min(b[1], c[1] - o[0]),
                     max(b[2], c[2] - o[1]), min(b[3], c[3] - o[1])]
        box[v.id] = tuple(b)
    b = [0, SIDE - 1, 0, SIDE - 1]
    for a, o in lane.targets.values():
        c = box[a]
        b = [max(b[0], c[0] - o[0]), min(b[1], c[1] - o[0]),
             max(b[2], c[2] - o[1]), min(b[3], c[3] - o[1])]
    for t in stores:
        if k.nodes[t].ctype is not CType.Int:
            return None
    for op, t in reduces:
        if op is not ReduceOp.Sum or k.nodes[t].ctype is not CType.Int:
            return None
    plan = BitPlan(lane, top, const, (b[0], b[1]), (b[2], b[3]))
    if not 16 <= plan.width <= lane.width or plan.height < 16:
        return None
    return plan


class BitEmitter:
    """Device code of the square: values are lists of planes, a plane a pair of C expressions
    (the words of columns 0-31 and 32-63) or False / True where it is all zeros / ones."""

    def __init__(self, plan: BitPlan, load_ptr):
        self.p, self.load_ptr = plan, load_ptr
        self.out: List[str] = []
        self.count = 0
        self.moved: Dict[tuple, tuple] = {}

    def new(self, e0: str, e1: str):
        self.count += 1
        self.out.append("const unsigned q%d_0 = %s, q%d_1 = %s;" % (self.count, e0, self.count, e1))
        return ("q%d_0" % self.count, "q%d_1" % self.count)

    # ------------------------------------------------------------ planes
    def neg(self, a):
        return (not a) if isinstance(a, bool) else self.new("~%s" % a[0], "~%s" % a[1])

    def both(self, a, b):
        if a is False or b is False:
            return False
        if a is True or b is True:
            return b if a is True else a
        return self.new(*("%s & %s" % x for x in zip(a, b)))

    def either(self, a, b):
        if a is True or b is True:
            return True
        if a is False or b is False:
            return b if a is False else a
        return self.new(*("%s | %s" % x for x in zip(a, b)))

    def differ(self, a, b):
        if isinstance(a, bool) or isinstance(b, bool):
            c, x = (a, b) if isinstance(a, bool) else (b, a)
            return self.neg(x) if c else x
        return self.new(*("%s ^ %s" % x for x in zip(a, b)))

    def major(self, a, b, c):
        xs = sorted((a, b, c), key=lambda x: not isinstance(x, bool))
        if isinstance(xs[0], bool):
            return self.either(xs[1], xs[2]) if xs[0] else self.both(xs[1], xs[2])
        return self.three(a, b, c, 0xe8)

    def three(self, a, b, c, table: int):
        """Any function of three bits in one instruction (its truth table, a the high bit)."""
        return self.new(*("__builtin_amdgcn_bitop3_b32(%s, %s, %s, %d)" % (x, y, z, table)
                          for x, y, z in zip(a, b, c)))

    def odd(self, a, b, c):
        if any(isinstance(x, bool) for x in (a, b, c)):
            return self.differ(self.differ(a, b), c)
        return self.three(a, b, c, 0x96)

    def choose(self, c, a, b):
        if isinstance(c, bool):
            return a if c else b
        if isinstance(a, bool) or isinstance(b, bool):
            return self.either(self.both(c, a), self.both(self.neg(c), b))
        return self.three(c, a, b, 0xca)

    def shift(self, key, plane, dx, dy):
        """The plane read at (dx, dy)."""
        if isinstance(plane, bool) or (dx == 0 and dy == 0):
            return plane
        if key + (dx, dy) in self.moved:
            return self.moved[key + (dx, dy)]
        if dy:
            p = self.shift(key, plane, 0, 0) if dx == 0 else self.shift(key, plane, 0, dy)
            if dx == 0:
                got = self.new(*("(unsigned)om_lane<%d>((int)%s)" % (dy, w) for w in plane))
                self.moved[key + (dx, dy)] = got
                return got
            plane = p
        if dx > 0:
            got = self.new("__builtin_amdgcn_alignbit(%s, %s, %d)" % (plane[1], plane[0], dx),
                           "%s >> %d" % (plane[1], dx))
        else:
            got = self.new("%s << %d" % (plane[0], -dx),
                           "__builtin_amdgcn_alignbit(%s, %s, %d)" % (plane[1], plane[0], 32 + dx))
        self.moved[key + (dx, dy)] = got
        return got

    # ------------------------------------------------------------ values
    def total(self, numbers: List[list]) -> list:
        """The sum of numbers (lists of planes): carry-save adders, weight by weight."""
        cols: List[list] = []
        for x in numbers:
            for i, plane in enumerate(x):
                while len(cols) <= i:
                    cols.append([])
                if plane is not False:
                    cols[i].append(plane)
        out, i = [], 0
        while i < len(cols):
            c = cols[i]
            if i + 1 == len(cols) and len(c) > 1:
                cols.append([])
            while len(c) > 2:
                a, b, d = c[:3]
                c[:3] = [self.odd(a, b, d)]
                c.append(c.pop(0))
                cols[i + 1].append(self.major(a, b, d))
            if len(c) == 2:
                a, b = c
                cols[i + 1].append(self.both(a, b))
                c[:] = [self.differ(a, b)]
            out.append(c[0] if c else False)
            i += 1
        return out

    def at_most(self, x: list, c: int):
        """x <= c"""
        if c < 0:
            return False
        if c >= (1 << len(x)) - 1:
            return True
        less, equal = False, True
        for i in reversed(range(len(x))):
            if c >> i & 1:
                less = self.either(less, self.both(equal, self.neg(x[i])))
                equal = self.both(equal, x[i])
            else:
                equal = self.both(equal, self.neg(x[i]))
        return self.either(less, equal)

    def equals(self, x: list, c: int):
        if c < 0 or c >> len(x):
            return False
        r = True
        for i, plane in enumerate(x):
            r = self.both(r, plane if c >> i & 1 else self.neg(plane))
        return r

    def compare(self, op: Op, x: list, c: int):
        if op is Op.EQ:
            return self.equals(x, c)
        if op is Op.NE:
            return self.neg(self.equals(x, c))
        if op is Op.LE:
            return self.at_most(x, c)
        if op is Op.LT:
            return self.at_most(x, c - 1)
        return self.neg(self.at_most(x, c - 1 if op is Op.GE else c))

    def evaluate(self, loads: Dict[int, tuple]) -> Dict[int, list]:
        """Planes of every value, from those of the loads."""
        p = self.p
        val: Dict[int, list] = {}
        users: Dict[int, int] = {}
        by_id = {v.id: v for v in p.lane.values}
        for v in p.lane.values:
            for b, o in v.args:
                if o is not None:
                    users[b] = users.get(b, 0) + 1
        for b, _ in p.lane.targets.values():
            users[b] = users.get(b, 0) + 2

        def digits(c):
            return [bool(c >> i & 1) for i in range(max(1, c.bit_length()))]

        def arg(b, o):
            if o is None:
                return digits(p.const[b])
            return [self.shift((b, i), plane, o[0], o[1]) for i, plane in enumerate(val[b])]

        def terms(v):
            """The numbers a chain of additions adds up (inner sums that nothing else reads)."""
            out = []
            for b, o in v.args:
                w = by_id.get(b) if o is not None else None
                if (w is not None and w.op == "arith" and w.payload[0] is Op.Add
                        and users[b] == 1 and not any(o)):
                    out += terms(w)
                else:
                    out.append((b, o))
            return out
        inner = set()
        for v in p.lane.values:
            if v.op == "arith" and v.payload[0] is Op.Add:
                for b, o in v.args:
                    if o is not None and not any(o) and users[b] == 1 and by_id[b].op == "arith" \
                            and by_id[b].payload[0] is Op.Add:
                        inner.add(b)
        for v in p.lane.values:
            if v.id in inner:
                continue
            if v.op == "load":
                val[v.id] = [loads[v.payload]]
                continue
            op = v.payload[0]
            if op is Op.Add:
                x = self.total([arg(b, o) for b, o in terms(v)])
                val[v.id] = x[:max(1, p.top[v.id].bit_length())]
            elif op in COMPARISONS:
                (b0, o0), (b1, o1) = v.args
                if o0 is None:               # constant first: mirror
                    op = {Op.LT: Op.GT, Op.GT: Op.LT, Op.LE: Op.GE, Op.GE: Op.LE}.get(op, op)
                    (b0, o0), (b1, o1) = v.args[1], v.args[0]
                val[v.id] = [self.compare(op, arg(b0, o0), p.const[b1])]
            elif op is Op.Not:
                val[v.id] = [self.neg(arg(*v.args[0])[0])]
            elif op in (Op.And, Op.Or):
                a, b = (arg(*x)[0] for x in v.args)
                val[v.id] = [self.both(a, b) if op is Op.And else self.either(a, b)]
            else:
                c, x, y = (arg(*z) for z in v.args)
                n = max(1, p.top[v.id].bit_length())
                x, y = (z + [False] * (n - len(z)) for z in (x, y))
                val[v.id] = [self.choose(c[0], x[i], y[i]) for i in range(n)]
        return val

    def word(self, plane) -> Tuple[str, str]:
        return plane if not isinstance(plane, bool) else (("~0u",) * 2 if plane else ("0u",) * 2)

    def body(self, stores, reduces) -> List[str]:
        """The square of the wave: ``stores`` (C pointer, C type, target), ``reduces``
        (accumulator, target); the caller has read the loads into l<static>_0 and _1."""
        p = self.p
        loads = {v.payload: ("l%d_0" % v.payload, "l%d_1" % v.payload)
                 for v in p.lane.values if v.op == "load"}
        val = self.evaluate(loads)

        def target(t):
            b, o = p.lane.targets[t]
            return [self.shift((b, i), plane, o[0], o[1]) for i, plane in enumerate(val[b])]
        w = self.out.append
        (c0, c1), (r0, r1) = p.cols, p.rows
        for acc, t in reduces:
            planes = [self.word(x) for x in target(t)]
            w("if (lane >= %d && lane <= %d && S0 + lane - %d < a.n1) {" % (r0, r1, r0))
            for i, (w0, w1) in enumerate(planes):
                w("  %s += (int)((unsigned)(__popc(%s & m0) + __popc(%s & m1)) << %d);"
                  % (acc, w0, w1, i))
            w("}")
        results = [(ptr, tn, [self.word(x) for x in target(t)]) for ptr, tn, t in stores]
        w("#pragma unroll 8")
        w("for (int r = 0; r < %d; ++r) {" % p.height)
        w("  if (S0 + r >= a.n1) break;")
        for ptr, tn, planes in results:
            terms = []
            for i, (w0, w1) in enumerate(planes):
                w("  const unsigned long long p%d = (unsigned)__builtin_amdgcn_readlane((int)%s, r + %d) | "
                  "(unsigned long long)(unsigned)__builtin_amdgcn_readlane((int)%s, r + %d) << 32;"
                  % (i, w0, r0, w1, r0))
                terms.append("(__builtin_amdgcn_inverse_ballot_w64(p%d) ? %d : 0)" % (i, 1 << i))
            w("  if (ok) om_put(%s + (size_t)(S0 + r) * a.n0, x, (%s)(%s));" % (ptr, tn, " + ".join(terms)))
        w("}")
        return self.out

    def pack(self) -> List[str]:
        """The rows of the square, turned: l<static>_0 and _1 of lane r hold row r, ``bad`` is
        set in a lane that read anything but 0 or 1."""
        p, out = self.p, []
        r0 = p.rows[0]
        statics = sorted(v.payload for v in p.lane.values if v.op == "load")
        out.append("int bad = 0;")
        for s in statics:
            out.append("unsigned l%d_0 = 0, l%d_1 = 0;" % (s, s))
        # every load before the first ballot: one memory latency, not one per batch of rows
        out.append("const int xl = om_wrap(x, a.n0, a.wide);")
        for s in statics:
            out.append("int c%d[%d];" % (s, SIDE))
        # rows inside the grid are a stride apart, two scalar instructions each instead of six;
        # the turn is repeated in both branches, as joining them behind the loads would hold
        # 64 addresses in registers
        turn = ["#pragma unroll", "  for (int j = 0; j < %d; ++j) {" % SIDE]
        for s in statics:
            turn += ["    bad |= c%d[j];" % s,
                     "    om_turn(j, __ballot(c%d[j] != 0), l%d_0, l%d_1);" % (s, s, s)]
        turn.append("  }")
        out += ["if (S0 >= %d && S0 + %d <= a.n1) {" % (r0, SIDE - r0)]
        for s in statics:
            out.append("  const int* f%d = %s + (size_t)(S0 - %d) * a.n0;" % (s, self.load_ptr(s), r0))
        out += ["#pragma unroll", "  for (int j = 0; j < %d; ++j) {" % SIDE]
        for s in statics:
            out.append("    c%d[j] = om_at(f%d, xl); f%d += a.n0;" % (s, s, s))
        out += ["  }"] + turn + ["} else {", "  int y = om_wrap(S0 - %d, a.n1, a.wide);" % r0,
                "#pragma unroll", "  for (int j = 0; j < %d; ++j) {" % SIDE]
        for s in statics:
            out.append("    c%d[j] = om_at(%s + (size_t)y * a.n0, xl);" % (s, self.load_ptr(s)))
        out += ["    y = y + 1 == a.n1 ? 0 : y + 1;", "  }"] + turn + ["}"]
        return out

"""Lowered SSA form of one OM kernel for the HIP backend.

The OM graph (``OM/Graph.hs``) is bipartite and, because the Builder never
shares sub-expressions, full of duplicates.  The HIP backend first turns each
kernel into a compact SSA list of value operations with:

* value numbering (identical operation on identical arguments -> one value),
* exact constant folding (integers, booleans, and IEEE float operations done
  in the value's own precision with numpy, so folded bits equal run-time bits),
* a symbolic range analysis for ``LoadIndex``/``LoadSize`` on Cyclic axes:
  an index lies in ``[0, n-1]`` and the size is ``n``, which decides
  comparisons such as the out-of-domain test of a boundary condition.

Folding never changes results: every rewrite is value-preserving for all grid
sizes (IEEE operations are deterministic; comparisons are decided only when
they hold for every ``n >= 1``).

With ``exact=True`` (the fast FP32 builds) floating constants are instead
folded in exact rational arithmetic from the literals the program wrote and
rounded once: ``1.4 - 1`` becomes the binary32 nearest 2/5 rather than the
difference of the rounded 1.4 and 1, and ``1 / (1.4 - 1)`` becomes exactly 2.5.
The exact value of each floating constant is kept (``LKernel.exact``) so the
emitter can multiply by it with a compensated product.
"""
from __future__ import annotations

from dataclasses import dataclass, field
from fractions import Fraction
from typing import Dict, List, Optional, Tuple

import numpy as np

from ... import annotation as A
from ...om.arith import COMPARISONS, Op
from ...om.dyn import CType, Realm, fraction_to_float32, fraction_to_float64
from ...om.graph import (Arith, Broadcast, Graph, Imm, Load, LoadIndex, LoadSize,
                         Reduce, Shift, Store)


@dataclass
class LNode:
    id: int
    op: str                    # load imm index size shift arith reduce bcast
    args: Tuple[int, ...]
    realm: Realm
    ctype: CType
    payload: object = None     # static idx / literal / axis / vec / (Op, cast) / ReduceOp
    hint_manifest: bool = False
    om_nodes: List[int] = field(default_factory=list)

    @property
    def arith_op(self) -> Optional[Op]:
        return self.payload[0] if self.op == "arith" else None


@dataclass
class LKernel:
    name: str
    nodes: List[LNode]
    stores: List[Tuple[int, int]]           # (static idx, value id)
    ndim: int
    # exact rational value of each floating constant (exact-folding builds only)
    exact: Dict[int, Fraction] = field(default_factory=dict)

    def users(self) -> List[List[int]]:
        u = [[] for _ in self.nodes]
        for n in self.nodes:
            for a in n.args:
                u[a].append(n.id)
        return u


# ------------------------------------------------------------ range analysis
class _Rng:
    """Interval [lo, hi] with bounds k*n_axis + c (axis None: plain constants)."""
    __slots__ = ("axis", "lo", "hi")

    def __init__(self, axis, lo, hi):
        self.axis, self.lo, self.hi = axis, lo, hi


def _lt_always(a: _Rng, b: _Rng) -> Optional[bool]:
    """True if a < b for every n >= 1, False if a >= b for every n >= 1, else None."""
    if a.axis is not None and b.axis is not None and a.axis != b.axis:
        return None
    dk, dc = a.hi[0] - b.lo[0], a.hi[1] - b.lo[1]
    if dk <= 0 and dk + dc < 0:
        return True
    dk, dc = a.lo[0] - b.hi[0], a.lo[1] - b.hi[1]
    if dk >= 0 and dk + dc >= 0:
        return False
    return None


def _np_scalar(v, ct: CType):
    if ct is CType.Float:
        return np.float32(v)
    if ct is CType.Double:
        return np.float64(v)
    if ct is CType.Int:
        return np.int32(v)
    return bool(v)


def _fold(op: Op, vals, ct_args: List[CType], ct_out: CType, cast_to):
    """Exact evaluation of a pure operation on constants, or None."""
    with np.errstate(all="ignore"):
        a = [_np_scalar(v, c) for v, c in zip(vals, ct_args)]
        try:
            if op is Op.Add:
                r = a[0] + a[1]
            elif op is Op.Sub:
                r = a[0] - a[1]
            elif op is Op.Mul:
                r = a[0] * a[1]
            elif op is Op.Div:
                if ct_args[0] is CType.Int:
                    if int(a[1]) == 0:
                        return None
                    q = abs(int(a[0])) // abs(int(a[1]))
                    r = np.int32(q if (int(a[0]) >= 0) == (int(a[1]) >= 0) else -q)
                else:
                    r = a[0] / a[1]
            elif op is Op.Mod:
                if ct_args[0] is not CType.Int or int(a[1]) == 0:
                    return None
                q = abs(int(a[0])) % abs(int(a[1]))
                r = np.int32(q if int(a[0]) >= 0 else -q)
            elif op is Op.Neg:
                r = -a[0]
            elif op is Op.Inv:
                if not ct_args[0].is_float:
                    return None
                r = _np_scalar(1, ct_args[0]) / a[0]
            elif op is Op.Not:
                r = not a[0]
            elif op is Op.And:
                r = bool(a[0]) and bool(a[1])
            elif op is Op.Or:
                r = bool(a[0]) or bool(a[1])
            elif op in COMPARISONS:
                r = {Op.EQ: a[0] == a[1], Op.NE: a[0] != a[1], Op.LT: a[0] < a[1],
                     Op.LE: a[0] <= a[1], Op.GT: a[0] > a[1], Op.GE: a[0] >= a[1]}[op]
                r = bool(r)
            elif op is Op.Max:
                r = a[1] if a[0] < a[1] else a[0]          # std::max
            elif op is Op.Min:
                r = a[1] if a[1] < a[0] else a[0]          # std::min
            elif op is Op.Select:
                r = a[1] if a[0] else a[2]
            elif op is Op.Sqrt and ct_args[0].is_float:
                r = np.sqrt(a[0])
            elif op is Op.Cast:
                if cast_to is CType.Int:
                    r = np.int32(int(a[0]))
                elif cast_to is CType.Bool:
                    r = bool(a[0])
                else:
                    r = _np_scalar(a[0], cast_to)
            else:
                return None
        except (OverflowError, ValueError, ZeroDivisionError):
            return None
    return _np_scalar(r, ct_out) if ct_out is not CType.Bool else bool(r)


def round_exact(x: Fraction, ct: CType):
    """The value of type ``ct`` nearest the rational ``x`` (ties to even)."""
    return fraction_to_float32(x) if ct is CType.Float else np.float64(fraction_to_float64(x))


def _fold_exact(op: Op, xs: List[Fraction], ct_args: List[CType], cast_to) -> Optional[Fraction]:
    """Exact rational value of an operation on exact constants, or None."""
    try:
        if op is Op.Add:
            return xs[0] + xs[1]
        if op is Op.Sub:
            return xs[0] - xs[1]
        if op is Op.Mul:
            return xs[0] * xs[1]
        if op is Op.Div:
            return xs[0] / xs[1]
        if op is Op.Neg:
            return -xs[0]
        if op is Op.Inv:
            return 1 / xs[0]
        if op is Op.Cast and cast_to is not None and cast_to.is_float:
            return xs[0]
    except ZeroDivisionError:
        return None
    return None


# ------------------------------------------------------------ building
def lower_kernel(om, ki: int, cyclic: Tuple[bool, ...], exact: bool = False,
                 merge: bool = True) -> LKernel:
    """``exact``: fold floating constants in exact rational arithmetic (see above).
    ``merge``: compute what both sides of a Select compute alike once, after it
    (``merge_selects``)."""
    g: Graph = om.kernels[ki].graph
    nodes: List[LNode] = []
    memo: Dict[tuple, int] = {}
    val_map: Dict[int, int] = {}           # OM value id -> LNode id
    const: Dict[int, object] = {}
    xval: Dict[int, Fraction] = {}         # exact value of floating (and integer) constants
    rng: Dict[int, _Rng] = {}

    def emit(op, args, realm, ct, payload, om_id, hint=False) -> int:
        key = (op, args, realm, ct, _hashable(payload))
        if key in memo:
            nid = memo[key]
            nodes[nid].om_nodes.append(om_id)
            nodes[nid].hint_manifest |= hint
            return nid
        nid = len(nodes)
        nodes.append(LNode(nid, op, args, realm, ct, payload, hint, [om_id]))
        memo[key] = nid
        return nid

    def make_const(value, realm, ct, om_id, ex: Optional[Fraction] = None) -> int:
        v = _np_scalar(value, ct) if ct is not CType.Bool else bool(value)
        if exact and ct is not CType.Bool and ex is None:
            ex = Fraction(int(v)) if ct is CType.Int else Fraction(float(v))
        if exact and ct.is_float:
            # constants that round alike but differ exactly stay apart
            nid = emit("imm", (), realm, ct, (v, ex), om_id)
            nodes[nid].payload = v
        else:
            nid = emit("imm", (), realm, ct, v, om_id)
        const[nid] = v
        if ex is not None:
            xval[nid] = ex
        if ct is not CType.Bool:
            rng[nid] = _Rng(None, (0, v), (0, v))
        return nid

    stores = []
    for v, node in enumerate(g.nodes):
        if not node.is_value:
            if isinstance(node.inst, Store):
                stores.append((node.inst.static, val_map[g.pre(v)[0]]))
            continue
        _, inst = g.inst_of_value(v)
        inst_id = g.pre(v)[0]
        args = tuple(val_map[p] for p in g.pre(inst_id))
        realm, ct = node.dyn.realm, node.dyn.ctype
        hint = A.to_maybe(A.Allocation, node.anot) is A.Allocation.Manifest
        if isinstance(inst, Load):
            nid = emit("load", (), realm, ct, inst.static, v)
        elif isinstance(inst, Imm):
            ex = None
            if exact and ct.is_float and getattr(inst, "exact", None) is not None:
                ex = Fraction(inst.exact)
            nid = make_const(inst.value, realm, ct, v, ex)
        elif isinstance(inst, LoadIndex):
            nid = emit("index", (), realm, ct, inst.axis, v)
            if cyclic[inst.axis]:
                rng[nid] = _Rng(inst.axis, (0, 0), (1, -1))
        elif isinstance(inst, LoadSize):
            nid = emit("size", (), realm, ct, inst.axis, v)
            rng[nid] = _Rng(inst.axis, (1, 0), (1, 0))
        elif isinstance(inst, Shift):
            if args[0] in const:
                nid = make_const(const[args[0]], realm, ct, v, xval.get(args[0]))
            elif all(x == 0 for x in inst.vec):
                nid = args[0]
                nodes[nid].om_nodes.append(v)
            else:
                nid = emit("shift", args, realm, ct, inst.vec, v)
        elif isinstance(inst, Broadcast):
            if args[0] in const:
                nid = make_const(const[args[0]], realm, ct, v, xval.get(args[0]))
            else:
                nid = emit("bcast", args, realm, ct, None, v)
                if args[0] in rng:
                    rng[nid] = rng[args[0]]
        elif isinstance(inst, Reduce):
            nid = emit("reduce", args, realm, ct, inst.op, v)
        elif isinstance(inst, Arith):
            op = inst.op
            nid = None
            if (exact and ct.is_float and args and all(a in xval for a in args)
                    and all(nodes[a].ctype is not CType.Bool for a in args)):
                ex = _fold_exact(op, [xval[a] for a in args], [nodes[a].ctype for a in args],
                                 inst.cast_to)
                if ex is not None:
                    nid = make_const(round_exact(ex, ct), realm, ct, v, ex)
            if nid is None and all(a in const for a in args):
                r = _fold(op, [const[a] for a in args], [nodes[a].ctype for a in args], ct,
                          inst.cast_to)
                if r is not None:
                    nid = make_const(r, realm, ct, v)
            if nid is None and exact and ct.is_float and op in (Op.Add, Op.Sub, Op.Mul):
                # x * 0, x * 1, x + 0 and x - 0 of finite operands (the sign of a zero
                # result aside): e.g. the pressure term p * delta(i, j) of an off-diagonal
                # momentum flux, Hydro.hs:113-114
                x0, x1 = xval.get(args[0]), xval.get(args[1])
                if op is Op.Mul and 0 in (x0, x1):
                    nid = make_const(0, realm, ct, v, Fraction(0))
                elif op is Op.Mul and (x0 == 1 or x1 == 1):
                    nid = args[1] if x0 == 1 else args[0]
                elif op is Op.Add and (x0 == 0 or x1 == 0):
                    nid = args[1] if x0 == 0 else args[0]
                elif op is Op.Sub and x1 == 0:
                    nid = args[0]
                if nid is not None and nid in (args[0], args[1]):
                    nodes[nid].om_nodes.append(v)
            if nid is None and op is Op.Select and args[0] in const:
                nid = args[1] if const[args[0]] else args[2]
                nodes[nid].om_nodes.append(v)
            if nid is None and op in (Op.And, Op.Or):
                for a, b in ((args[0], args[1]), (args[1], args[0])):
                    if a in const:
                        if (op is Op.And and not const[a]) or (op is Op.Or and const[a]):
                            nid = make_const(const[a], realm, ct, v)
                        else:
                            nid = b
                            nodes[nid].om_nodes.append(v)
                        break
            if nid is None and op in COMPARISONS and args[0] in rng and args[1] in rng:
                ra, rb = rng[args[0]], rng[args[1]]
                dec = None
                if op is Op.LT:
                    dec = _lt_always(ra, rb)
                elif op is Op.GE:
                    d = _lt_always(ra, rb)
                    dec = None if d is None else (not d)
                elif op is Op.GT:
                    dec = _lt_always(rb, ra)
                elif op is Op.LE:
                    d = _lt_always(rb, ra)
                    dec = None if d is None else (not d)
                if dec is not None:
                    nid = make_const(dec, realm, ct, v)
            if nid is None:
                nid = emit("arith", args, realm, ct, (op, inst.cast_to), v, hint)
                if op is Op.Cast and args[0] in rng and inst.cast_to is not CType.Bool:
                    rng[nid] = rng[args[0]]
        else:
            raise TypeError(inst)
        val_map[v] = nid
    fx = {n: x for n, x in xval.items() if nodes[n].ctype.is_float}
    k = _prune(LKernel(om.kernels[ki].name, nodes, stores, om.ndim, fx))
    return merge_selects(k) if merge else k


# What an operation costs next to an addition, where merge_selects weighs the operations it
# saves against the selects it adds: a division or root is a reciprocal or root instruction at
# a quarter of the rate and a multiply (far more where it is correctly rounded).
_WEIGHT = {Op.Div: 5, Op.Inv: 4, Op.Sqrt: 4, Op.Exp: 20, Op.Log: 20, Op.Sin: 20, Op.Cos: 20,
           Op.Tan: 20, Op.Asin: 20, Op.Acos: 20, Op.Atan: 20, Op.Atan2: 40, Op.Pow: 40}


def merge_selects(k: LKernel) -> LKernel:
    """Select first, compute once.

    ``c ? f(a) : f(b)`` is ``f(c ? a : b)``: the same operation on the value the condition
    picks, so the results are the same bits, and one evaluation of f is saved.  HLLC selects
    between the fluxes of four states after computing all of them (Hydro's ``selector``): with
    the two star states behind one select, a face evaluates one star state and its flux.

    The reference's selector is a chain, ``c1 ? a : (c2 ? b : (c3 ? c : d))``, in which the two
    alike (b and c) do not meet in one Select.  It is first rewritten as ``(c1 || (!c2 &&
    !c3)) ? (c1 ? a : d) : (c2 ? b : c)``, which picks the same operand for every value of the
    three conditions.

    The Hydro step falls from 779 to 685 operations per cell.  Measured: 2048^2 FP32 124 -> 110
    us per step, 1024^2 FP64 99 -> 86 us (same bits), 256 uneven grids 0.998 -> 0.888 ms.

    A group is merged only where it costs less: what it saves is the operations that nothing
    else reads, what it adds is a Select per input that differs."""
    nodes = list(k.nodes)
    stores = list(k.stores)
    memo = {(n.op, n.args, n.realm, n.ctype, _hashable(n.payload)): n.id for n in nodes
            if n.op == "arith"}

    def add(op, args, realm, ct, cast_to=None, like=None) -> int:
        payload = (op, cast_to)
        key = ("arith", tuple(args), realm, ct, _hashable(payload))
        if key not in memo:
            memo[key] = len(nodes)
            nodes.append(LNode(len(nodes), "arith", tuple(args), realm, ct, payload, False,
                               list(like.om_nodes) if like is not None else []))
        return memo[key]

    def is_select(v):
        return nodes[v].op == "arith" and nodes[v].payload[0] is Op.Select

    def users_of():
        u: Dict[int, List[int]] = {n.id: [] for n in nodes}
        live = _reach(nodes, [v for _, v in stores])
        for n in nodes:
            if n.id in live:
                for a in n.args:
                    u[a].append(n.id)
        return u, live

    def replace(new: Dict[int, int]):
        """Point every reader of a key at its value (stores too)."""
        for n in nodes:
            if any(a in new for a in n.args):
                n.args = tuple(new.get(a, a) for a in n.args)
        stores[:] = [(s, new.get(v, v)) for s, v in stores]

    nodes = [LNode(n.id, n.op, n.args, n.realm, n.ctype, n.payload, n.hint_manifest,
                   list(n.om_nodes)) for n in nodes]
    # ---- chains
    users, live = users_of()
    stored = set(v for _, v in stores)
    alone = lambda v: len(users[v]) == 1 and v not in stored

    def alike(x, y):
        a, b = nodes[x], nodes[y]
        return (a.op == "arith" and b.op == "arith" and a.payload == b.payload
                and a.ctype is b.ctype and len(a.args) == len(b.args) and x != y)
    new: Dict[int, int] = {}
    for s1 in sorted(live):
        if not is_select(s1) or nodes[s1].realm is not Realm.Array:
            continue
        c1, a, s2 = nodes[s1].args
        if not is_select(s2) or not alone(s2):
            continue
        c2, b, s3 = nodes[s2].args
        if not is_select(s3) or not alone(s3):
            continue
        c3, c, d = nodes[s3].args
        if not alike(b, c) or is_select(b):
            continue
        n = nodes[s1]
        R = n.realm
        neither = add(Op.And, (add(Op.Not, (c2,), R, CType.Bool), add(Op.Not, (c3,), R, CType.Bool)),
                      R, CType.Bool)
        outer = add(Op.Or, (c1, neither), R, CType.Bool)
        out = add(Op.Select, (outer, add(Op.Select, (c1, a, d), R, n.ctype, like=n),
                              add(Op.Select, (c2, b, c), R, n.ctype, like=n)), R, n.ctype, like=n)
        nodes[out].hint_manifest |= n.hint_manifest
        new[s1] = out
    replace(new)
    changed = bool(new)
    # ---- groups of selects with one condition
    done = set()
    while True:
        users, live = users_of()
        stored = set(v for _, v in stores)
        groups: Dict[int, List[int]] = {}
        for v in sorted(live):
            if is_select(v) and nodes[v].realm is Realm.Array:
                groups.setdefault(nodes[v].args[0], []).append(v)
        todo = [c for c in groups if c not in done]
        if not todo:
            break
        cond = todo[0]
        done.add(cond)
        sels = groups[cond]
        selset = set(sels)
        # operations that only these selects read, directly or through each other
        only: set = set()
        for v in _topological(nodes, live)[::-1]:
            n = nodes[v]
            if n.op != "arith" or v in stored or v in selset or n.hint_manifest or not users[v]:
                continue
            if all((u in only) or (u in selset and nodes[u].args[0] != v) for u in users[v]):
                only.add(v)
        pairs: Dict[Tuple[int, int], Optional[Tuple]] = {}

        def visit(x, y):
            """Plan the merged value of the pair: None for a Select, else its argument pairs."""
            if x == y or (x, y) in pairs:
                return
            if x in only and y in only and alike(x, y):
                pairs[(x, y)] = tuple(zip(nodes[x].args, nodes[y].args))
                for p in pairs[(x, y)]:
                    visit(*p)
            else:
                pairs[(x, y)] = None
        for s in sels:
            visit(*nodes[s].args[1:])
        weight = lambda v: _WEIGHT.get(nodes[v].payload[0], 1)
        gone = set(z for p, q in pairs.items() if q is not None for z in p)
        saved = sum(weight(v) for v in gone) + len(sels)
        spent = sum(1 if q is None else weight(p[0]) for p, q in pairs.items())
        if not gone or spent >= saved:
            continue
        merged: Dict[Tuple[int, int], int] = {}

        def build(x, y):
            if x == y:
                return x
            if (x, y) not in merged:
                n = nodes[x]
                q = pairs[(x, y)]
                if q is None:
                    merged[(x, y)] = add(Op.Select, (cond, x, y), n.realm, n.ctype, like=n)
                else:
                    merged[(x, y)] = add(n.payload[0], tuple(build(*p) for p in q), n.realm,
                                         n.ctype, n.payload[1], like=n)
            return merged[(x, y)]
        new = {}
        for s in sels:
            m = build(*nodes[s].args[1:])
            if m != s:
                nodes[m].hint_manifest |= nodes[s].hint_manifest
                new[s] = m
        replace(new)
        changed |= bool(new)
    if not changed:
        return k
    order = _topological(nodes, _reach(nodes, [v for _, v in stores]))
    at = {v: i for i, v in enumerate(order)}
    out = [LNode(at[v], nodes[v].op, tuple(at[a] for a in nodes[v].args), nodes[v].realm,
                 nodes[v].ctype, nodes[v].payload, nodes[v].hint_manifest, nodes[v].om_nodes)
           for v in order]
    return LKernel(k.name, out, [(s, at[v]) for s, v in stores], k.ndim,
                   {at[n]: x for n, x in k.exact.items() if n in at})


def _reach(nodes, roots) -> set:
    seen, stack = set(), list(roots)
    while stack:
        x = stack.pop()
        if x not in seen:
            seen.add(x)
            stack.extend(nodes[x].args)
    return seen


def _topological(nodes, live) -> List[int]:
    """The live values, every one after its arguments, otherwise in numbering order."""
    out, state = [], {}
    for root in sorted(live):
        stack = [root]
        while stack:
            x = stack[-1]
            if state.get(x) == 2:
                stack.pop()
                continue
            state[x] = 1
            wait = [a for a in nodes[x].args if state.get(a) != 2]
            if wait:
                stack.extend(reversed(wait))
            else:
                state[x] = 2
                out.append(x)
                stack.pop()
    return out


def _hashable(p):
    if isinstance(p, np.generic):
        return (type(p).__name__, p.tobytes())
    return p


def _prune(k: LKernel) -> LKernel:
    """Drop values no store reaches; renumber densely (topological order kept)."""
    live = set()
    stack = [v for _, v in k.stores]
    while stack:
        x = stack.pop()
        if x in live:
            continue
        live.add(x)
        stack.extend(k.nodes[x].args)
    remap = {}
    out = []
    for n in k.nodes:
        if n.id in live:
            remap[n.id] = len(out)
            out.append(LNode(len(out), n.op, tuple(remap[a] for a in n.args), n.realm, n.ctype,
                             n.payload, n.hint_manifest, n.om_nodes))
    return LKernel(k.name, out, [(s, remap[v]) for s, v in k.stores], k.ndim,
                   {remap[n]: x for n, x in k.exact.items() if n in remap})

"""Planning of box kernels: group kernels whose tiles have constant shapes.

``GroupPlan`` sizes every stage's region per tile at run time: exact, but a
tile then carries a region program, every sweep carries range checks and a
per-point path for the blocks a region's edge cuts, and every index depends
on run-time bounds.  For the 26 stages of a camera pipeline that was more
scalar than vector work (522 M scalar against 491 M vector instructions per
48-frame batch).

When the tile grid starts at constants and every access is a monotone map of
one variable with constant coefficients, each stage's region is instead a
box at ``A * tile + lo .. A * tile + hi`` with integer constants, the same
in every tile.  A ``BoxPlan`` holds those boxes.  The kernel
(``box_emit``) computes the whole box in every tile, so item counts, LDS
layouts and all index offsets are compile-time constants, and blocks need no
partial form: points past a box's end are computed from whatever the
(padded) LDS rows hold and never read by a point that counts.  Tiles whose
boxes lie inside every domain, Case and array run without any check; the
others clamp their global reads and check Cases and the output's range per
point.

Per-thread blocks are aligned to the parity their stage's expressions use:
with 2 x 2 blocks on even coordinates, ``x % 2 == 0`` and ``x / 2`` of an
upsampling or an interleave are known for each point of the block, so the
selects and divisions disappear, neighbouring points share their reads, and
lanes of one wavefront no longer disagree on the branch.

That also makes stages free whose definition only relabels other stages
(deinterleaving, colour planes, interleaving): they are substituted into
their readers (``_alias_inline``) and no longer pass through LDS.
"""

from fractions import Fraction

from .analysis import PlanError, Part, classify_access, ceval_int, eval_bexpr
from .constructs import Reference, Variable
from .cprint import same_expr
from .expr_ast import (AbstractBinaryOpNode, AbstractUnaryOpNode, Value, Parameter,
                       Condition, Select, Cast, InbuiltFunction)
from .expr_types import Int
from .expression import substitute_vars, substitute_refs, getType, _rebuild_bin
from .group_plan import GroupPlan, StageInfo

# gpu options that ask for a particular form of the general kernel
GENERAL_ONLY = ('block', 'block_lds', 'lanes', 'stage', 'no_inline', 'no_fuse', 'index64',
                'no_offset_inline', 'vlds')
MAX_POINTS = 16         # points of one per-thread block (registers)


def resident(threads, lds):
    """Workgroups a compute unit holds, by threads and bytes of LDS."""
    return min(2048 // threads, (160 * 1024) // max(1, lds))


def _has_param(e):
    return any(isinstance(v, Parameter) for v in e.collect(Variable)) if hasattr(e, 'collect') else False


def const_int(e):
    """The integer value of a bound without parameters, else None."""
    if e is None:
        return None
    try:
        return int(eval_bexpr(e, {}))
    except (PlanError, KeyError, AttributeError, TypeError):
        return None


# ---------------------------------------------------------------------------
# accesses
# ---------------------------------------------------------------------------

class Map(object):
    """One reference argument as a function of the consumer's point.

    kind 'const': ``value``.
    kind 'var':   f(x) of consumer dimension ``dim``; f(x + period) ==
                  f(x) + slope * period; ``f`` evaluates it with floor
                  division (equal to C's on the coordinates that count).
                  ``lows``/``highs``: bounds it is clamped to outside its
                  range (edge replication), [] if none.
    kind '*':     data dependent."""

    def __init__(self, kind, value=None, dim=None, slope=None, period=1, f=None, lows=(), highs=()):
        self.kind = kind
        self.value = value
        self.dim = dim
        self.slope = slope
        self.period = period
        self.f = f
        self.lows = list(lows)
        self.highs = list(highs)


def _divisors(e):
    """Product of the divisors in an index expression, and its numerators."""
    n, nums = 1, []
    stack = [e]
    while stack:
        x = Value.numericToValue(stack.pop())
        if isinstance(x, AbstractBinaryOpNode):
            if x.op == '/':
                n *= int(ceval_int(x.right, {}))
                nums.append(x.left)
            stack += [x.left, x.right]
        elif hasattr(x, 'children'):
            stack += list(x.children())
    return n, nums


def _strip_clamp(e):
    """(core, lower bounds, upper bounds) of ``Min(Max(core, lo), hi)`` in
    any nesting, the bounds free of variables; None when e is not one."""
    lows, highs = [], []
    e = Value.numericToValue(e)
    while isinstance(e, Select):
        c = e.condition
        if c.conditional not in ('>', '<') or not same_expr(c.lhs, e.true_expression) or \
                not same_expr(c.rhs, e.false_expression):
            return None
        l, r = Value.numericToValue(e.true_expression), Value.numericToValue(e.false_expression)

        def free(x):
            return not any(type(v) is Variable for v in x.collect(Variable)) and not x.has(Reference)
        if free(r):
            core, b = l, r
        elif free(l):
            core, b = r, l
        else:
            return None
        (lows if c.conditional == '>' else highs).append(b)
        e = core
    return (e, lows, highs) if lows or highs else None


def arg_map(arg, cvars):
    """``Map`` of a reference argument; PlanError when it depends on a
    parameter (its offset is then no constant)."""
    a = Value.numericToValue(arg)
    lows = highs = ()
    cl = _strip_clamp(a)
    if cl is not None:
        a, lows, highs = cl
    acc = classify_access(a, cvars)
    if acc.kind == '*' or (acc.kind == 'const' and cl is not None):
        return Map('*')
    if acc.kind == 'const':
        v = const_int(a)
        if v is None:
            raise PlanError("parameter in an index")
        return Map('const', value=v)
    if _has_param(a):
        raise PlanError("parameter in an index")
    if not acc.increasing:
        return Map('*')
    var, slope = acc.var, Fraction(acc.slope)
    per, _ = _divisors(a)
    if per > 64:
        return Map('*')
    big = per << 20

    def f(x):
        return ceval_int(a, {var: x + big}) - int(slope * big)
    return Map('var', dim=acc.dim, slope=slope, period=per, f=f, lows=lows, highs=highs)


class Span(object):
    """Coordinates ``A * t_d + lo .. A * t_d + hi`` (d None: constants)."""

    def __init__(self, d, A, lo, hi):
        self.d = d if A else None
        self.A = A
        self.lo = lo
        self.hi = hi

    def hull(self, o):
        if o is None:
            return self
        if (self.d, self.A) != (o.d, o.A):
            raise PlanError("an axis moves with two tile dimensions")
        return Span(self.d, self.A, min(self.lo, o.lo), max(self.hi, o.hi))

    @property
    def ext(self):
        return self.hi - self.lo + 1

    def key(self):
        return (self.d, self.A, self.lo, self.hi)


def image(m, span):
    """Span of a 'var' map over a span of its variable."""
    a = m.slope * span.A
    if a.denominator != 1 or (span.A and span.A % m.period):
        raise PlanError("a tile is no whole number of coarse points")
    return Span(span.d, int(a), m.f(span.lo), m.f(span.hi))


# ---------------------------------------------------------------------------
# expressions of one point of a block
# ---------------------------------------------------------------------------

class Known(object):
    """What is known of a stage's variables at one point of a block:
    ``value[v]`` an integer, or ``mod[v]`` = (modulus, residue); ``least[v]``
    a lower bound of v over the points that count (``least_values``)."""

    def __init__(self, value, mod, least=None):
        self.value = value
        self.mod = mod
        self.least = least or {}


def least_values(func, part):
    """{variable: constant lower bound} over the points of a Case part."""
    out = {}
    for v, dom, (lo, _) in zip(func.variables, func.domain, part.box):
        bounds = [b for b in (const_int(dom.lowerBound), const_int(lo)) if b is not None]
        if bounds:
            out[v] = max(bounds)
    return out


def _ival(e):
    return e.value if isinstance(e, Value) and isinstance(e.value, int) and \
        not isinstance(e.value, bool) else None


def decide(c, kn):
    """True, False or None (not known) for a condition whose sides fold."""
    if c.conditional in ('&&', '||'):
        l, r = decide(c.lhs, kn), decide(c.rhs, kn)
        if c.conditional == '&&':
            return False if (l is False or r is False) else (True if (l and r) else None)
        return True if (l or r) else (False if (l is False and r is False) else None)
    l, r = _ival(fold(c.lhs, kn)), _ival(fold(c.rhs, kn))
    if l is None or r is None:
        return None
    return {'==': l == r, '!=': l != r, '<': l < r, '<=': l <= r, '>': l > r, '>=': l >= r}[c.conditional]


def _shifted(e):
    """(variable, c) of an expression v + c, else None."""
    e = Value.numericToValue(e)
    if isinstance(e, Variable):
        return e, 0
    if isinstance(e, AbstractBinaryOpNode) and e.op in ('+', '-'):
        l, r = Value.numericToValue(e.left), Value.numericToValue(e.right)
        if _ival(r) is not None:
            m = _shifted(l)
            return m and (m[0], m[1] + (r.value if e.op == '+' else -r.value))
        if e.op == '+' and _ival(l) is not None:
            m = _shifted(r)
            return m and (m[0], m[1] + l.value)
    return None


def _residue(e, kn):
    """(modulus, residue) of an expression v + c that is nowhere negative
    (C's remainder of a negative number is negative), else None."""
    vc = _shifted(e)
    if vc is None or vc[0] not in kn.mod or kn.least.get(vc[0], -vc[1] - 1) + vc[1] < 0:
        return None
    m, r = kn.mod[vc[0]]
    return m, (r + vc[1]) % m


def fold(e, kn):
    """``e`` with what ``kn`` decides folded: variables of known value,
    remainders of known residue, integer arithmetic of constants, and
    selects whose condition is known (the taken branch with the casts a
    select applies).  Floating-point arithmetic is left alone."""
    e = Value.numericToValue(e)
    if isinstance(e, Variable) and not isinstance(e, Parameter):
        return Value(kn.value[e], Int) if e in kn.value else e
    if isinstance(e, (Value, Variable)):
        return e
    if isinstance(e, AbstractBinaryOpNode):
        if e.op == '%':
            m = _ival(Value.numericToValue(e.right))
            r = _residue(e.left, kn)
            if m and m > 0 and r and r[0] % m == 0:
                return Value(r[1] % m, Int)
        l, r = fold(e.left, kn), fold(e.right, kn)
        if _ival(l) is not None and _ival(r) is not None and e.op in ('+', '-', '*', '/', '%') and \
                not (e.op in '/%' and r.value == 0):
            # (a literal outside int makes C's arithmetic long long)
            v = ceval_int(_rebuild_bin(e, l, r), {})
            if all(-2 ** 31 <= i < 2 ** 31 for i in (v, l.value, r.value)):
                return Value(v, Int)
        return _rebuild_bin(e, l, r)
    if isinstance(e, AbstractUnaryOpNode):
        c = fold(e.child, kn)
        if _ival(c) is not None and e.op in ('-', '+'):
            return Value(-c.value if e.op == '-' else c.value, Int)
        return type(e)(c) if type(e) is not AbstractUnaryOpNode else AbstractUnaryOpNode(c, e.op)
    if isinstance(e, Reference):
        return Reference(e.objectRef, [fold(a, kn) for a in e.arguments])
    if isinstance(e, Cast):
        return Cast(e.typ, fold(e.expression, kn))
    if isinstance(e, Select):
        d = decide(e.condition, kn)
        if d is not None:
            t = e.true_expression if d else e.false_expression
            tt, te = getType(e), getType(Value.numericToValue(t))
            x = fold(t, kn)
            if not (isinstance(x, Reference) and x.objectRef.typ is te is tt):
                x = Cast(te, x)
                if te is not tt:
                    x = Cast(tt, x)
            return x
        return Select(fold_cond(e.condition, kn), _typed(fold(e.true_expression, kn), e.true_expression),
                      _typed(fold(e.false_expression, kn), e.false_expression), False)
    if isinstance(e, InbuiltFunction):
        return type(e)(*[fold(a, kn) for a in e.arguments])
    raise PlanError("cannot fold %s" % (e,))


def _typed(x, e):
    """x, folded from a select's branch e, with e's DSL type (a folded
    constant is an Int whatever its parts' types; a select's branches have
    one type)."""
    t = getType(Value.numericToValue(e))
    return x if getType(x) is t else Cast(t, x)


def fold_cond(c, kn):
    if c.conditional in ('&&', '||'):
        return Condition(fold_cond(c.lhs, kn), c.conditional, fold_cond(c.rhs, kn))
    return Condition(fold(c.lhs, kn), c.conditional, fold(c.rhs, kn))


def _mods(e, cvars, least):
    """[(dimension, modulus)] of the remainders in e that ``fold`` can know
    (``least``: ``least_values``)."""
    out = []
    stack = [e]
    while stack:
        x = Value.numericToValue(stack.pop())
        if isinstance(x, Condition):
            stack += [x.lhs, x.rhs]
            continue
        if isinstance(x, AbstractBinaryOpNode) and x.op == '%':
            m = _ival(Value.numericToValue(x.right))
            vc = _shifted(x.left)
            if m and vc and vc[0] in cvars and least.get(vc[0], -vc[1] - 1) + vc[1] >= 0:
                out.append((cvars.index(vc[0]), m))
        if isinstance(x, Select):
            stack += [x.condition, x.true_expression, x.false_expression]
        elif isinstance(x, Reference):
            stack += list(x.arguments)
        elif hasattr(x, 'children'):
            stack += list(x.children())
    return out


def _nops(e):
    """Operations of one point, reads and scaled reads aside."""
    n = 0
    stack = [e]
    while stack:
        x = Value.numericToValue(stack.pop())
        if isinstance(x, Condition):
            stack += [x.lhs, x.rhs]
            continue
        if isinstance(x, AbstractBinaryOpNode) and x.op == '*' and \
                any(isinstance(Value.numericToValue(a), Value) and
                    isinstance(Value.numericToValue(b), Reference)
                    for a, b in ((x.left, x.right), (x.right, x.left))):
            # a scaled read: neighbouring points share it (counted with the
            # read), or it is half of a fused multiply-add
            continue
        if isinstance(x, (AbstractBinaryOpNode, AbstractUnaryOpNode, Cast, Select)):
            n += 1
        elif isinstance(x, InbuiltFunction):
            n += 20
        if isinstance(x, Select):
            stack += [x.condition, x.true_expression, x.false_expression]
        elif isinstance(x, Reference):
            continue
        elif hasattr(x, 'children'):
            stack += list(x.children())
    return n


# ---------------------------------------------------------------------------
# the plan
# ---------------------------------------------------------------------------

class BoxPlan(GroupPlan):
    """Boxes, blocks and LDS layout of a box kernel; PlanError when the group
    has no constant boxes (the general kernel serves it then)."""

    @staticmethod
    def of(plan):
        """The box plan of a general plan's group, or None."""
        o = plan.opts
        if o.get('no_box') or any(o.get(k) for k in GENERAL_ONLY) or int(o.get('roll', 1)) > 1:
            return None
        def boxes(**opts):
            return BoxPlan(plan.pipe, plan.group, plan.gindex, plan.tile_sizes, dict(o, **opts))
        try:
            box = boxes()
            # LDS rows hold whole blocks, and the rows that pads cost can
            # halve the workgroups a compute unit holds: blocks of fewer rows
            # then, if they bring those back.  Harris, 16x512 tiles of 512
            # threads, 82.6 KB of LDS against 74.3 (general 74.3), us at
            # 1200x1600 / 2048x2048 / 3000x3000 / 4100x4100: 16.1 / 16.6 /
            # 31.3 / 55.6 with 4x2 blocks, 14.4 / 15.4 / 27.7 / 43.5 with
            # 2x2, general kernel 13.2 / 14.6 / 32.2 / 56.9.  (Two workgroups
            # instead of three are no reason: 16x340, w256, 11.9 / 18.9 / 31.9
            # / 51.5 against 12.6 / 19.1 / 29.9 / 47.9.)
            threads = int(o.get('threads', 256))
            want = resident(threads, plan.lds_bytes)
            for rows in (2, 1):
                if 2 * resident(threads, box.lds_bytes) > want:
                    break
                less = boxes(box_rows=rows)
                if resident(threads, less.lds_bytes) >= want:
                    box = less
            return box
        except PlanError:
            return None

    def _build(self, stage):
        comps = self.group.comps
        self.stages = [StageInfo(c, i) for i, c in enumerate(comps)]
        self.by_comp = dict((s.comp, s) for s in self.stages)
        liveouts = self.pipe.liveouts(self.group)
        for s in self.stages:
            s.liveout = s.comp in liveouts
        if sum(s.liveout for s in self.stages) != 1:
            raise PlanError("more than one live-out")
        if any(part.pred for s in self.stages for part in s.parts):
            raise PlanError("a Case with a predicate")
        self._offset_inline()
        self.aliases = []
        self._alias_inline()
        self._plane_inline()
        self._consumers()
        self._anchor()
        self._align()
        self._grid()
        self._inline()
        self._order()
        self._phases()
        self._boxes()
        self._layout()

    # -- substitutions -----------------------------------------------------------
    def _in_group_refs(self, p):
        """[(consumer, part, reference)] of the group's reads of stage p."""
        return [(c, cp, r) for c in self.stages for cp in c.parts for r in self._part_refs(cp)
                if r.objectRef is p.func]

    def _substitute(self, p, exprs):
        """Replace the reads of p by ``exprs`` (reference -> expression)."""
        for c in self.stages:
            parts = []
            for cp in c.parts:
                m = dict((r, exprs[id(r)]) for r in self._part_refs(cp) if id(r) in exprs)
                parts.append(Part(cp.box, cp.pred, substitute_refs(cp.expr, m), cp.case_index)
                             if m else cp)
            c.parts = parts
        self.stages.remove(p)
        self.by_comp = dict((s.comp, s) for s in self.stages)
        self.aliases.append(p.name)

    def _alias_inline(self):
        """Substitute stages that only relabel others into their readers.

        A stage whose value is a read (or a Select of reads on the parity of
        its own point, no arithmetic) costs nothing to evaluate: storing it
        is a pass over LDS and a barrier.  The camera pipeline's
        deinterleaving, its four colour planes and its interleaving are 14
        of 26 stages; each was one or two LDS reads and a write per point.
        Values keep the stage's type by a cast."""
        changed = True
        while changed:
            changed = False
            for p in self.stages:
                if p.liveout or not all(self._relabels(part.expr) for part in p.parts):
                    continue
                uses = self._in_group_refs(p)
                if not uses:
                    continue
                exprs = {}
                for (c, cp, r) in uses:
                    part = self._part_at(p, r)
                    if part is None or c is p:
                        exprs = None
                        break
                    body = substitute_vars(part.expr, dict(zip(p.func.variables, r.arguments)))
                    exprs[id(r)] = Cast(p.func.typ, body)
                if exprs:
                    self._substitute(p, exprs)
                    changed = True
                    break

    @staticmethod
    def _relabels(e):
        e = Value.numericToValue(e)
        if isinstance(e, Reference):
            return not any(a.has(Reference) for a in e.arguments if hasattr(a, 'has'))
        if type(e) is Select:
            stack = [e.condition]
            while stack:
                c = stack.pop()
                if c.conditional in ('&&', '||'):
                    stack += [c.lhs, c.rhs]
                elif any(Value.numericToValue(x).has(k) for x in (c.lhs, c.rhs)
                         for k in (Reference, Parameter)):
                    return False
            return BoxPlan._relabels(e.true_expression) and BoxPlan._relabels(e.false_expression)
        if isinstance(e, Cast):
            return e.typ is getType(e.expression) and BoxPlan._relabels(e.expression)
        return False

    @staticmethod
    def _part_at(p, r):
        """The one part of p that defines every point ``r`` can read: the
        only one whose constant bounds admit its constant arguments, the
        other dimensions unbounded; None when that cannot be said."""
        found = []
        for part in p.parts:
            ok = True
            for (lo, hi), a in zip(part.box, r.arguments):
                if lo is None and hi is None:
                    continue
                v = const_int(a) if not Value.numericToValue(a).has(Variable) else None
                l = const_int(lo) if lo is not None else -1 << 40
                h = const_int(hi) if hi is not None else 1 << 40
                if v is None or l is None or h is None:
                    return None
                ok = ok and l <= v <= h
            if ok:
                found.append(part)
        return found[0] if len(found) == 1 else None

    def _plane_inline(self):
        """Compute in its reader's registers a stage read only at the
        reader's own point and constant planes (``filtered`` reads
        ``interpolated(0, x, y)`` and ``(1, x, y)``): the planes share their
        loads and the LDS plane between the two goes away (bilateral: 60 KB
        of LDS per workgroup to 28 KB)."""
        for p in list(self.stages):
            if p.liveout or len(p.parts) != 1 or any(b != (None, None) for b in p.parts[0].box):
                continue
            uses = self._in_group_refs(p)
            if not uses or len(uses) > 4 or len(set(id(c) for (c, _, _) in uses)) != 1:
                continue
            c = uses[0][0]
            exprs = {}
            planes = False
            for (_, _, r) in uses:
                vs = []
                for a in r.arguments:
                    a = Value.numericToValue(a)
                    if _ival(a) is not None:
                        planes = True
                    else:
                        vs.append(a)
                own = [v for v in c.func.variables if any(v is x for x in vs)]
                if len(vs) != len(own) or not all(x is v for x, v in zip(vs, own)) or c is p:
                    exprs = None
                    break
                exprs[id(r)] = Cast(p.func.typ, substitute_vars(
                    p.parts[0].expr, dict(zip(p.func.variables, r.arguments))))
            if exprs and planes:
                self._substitute(p, exprs)

    def _order(self):
        """Every stage after the stages it reads."""
        done, out = set(), []

        def visit(s):
            if s in done:
                return
            done.add(s)
            for part in s.parts:
                for r in self._part_refs(part):
                    if self.in_group(r.objectRef):
                        visit(self.stage_of(r.objectRef))
            out.append(s)
        for s in self.stages:
            visit(s)
        self.stages = out

    # -- boxes and blocks ----------------------------------------------------------
    def _part_span(self, s, part, i):
        """s's span of dimension i cut to the part's bounds where both are
        constants; None when nothing is left."""
        sp = s.span[i]
        if sp.A:
            return sp
        lo, hi = const_int(part.box[i][0]), const_int(part.box[i][1])
        l = sp.lo if lo is None else max(sp.lo, lo)
        h = sp.hi if hi is None else min(sp.hi, hi)
        return Span(None, 0, l, h) if l <= h else None

    def _boxes(self):
        a = self.anchor
        tiled = dict(self.grid_dims)
        for s in reversed(self.stages):
            if s.nd == 0:
                raise PlanError("a stage without dimensions")
            for part in s.parts:
                for r in self._part_refs(part):
                    self._check_ref(s, r)
            if s is a:
                s.span = []
                for d in range(a.nd):
                    lb = const_int(a.func.domain[d].lowerBound)
                    ub = const_int(a.func.domain[d].upperBound)
                    if d in tiled:
                        if lb is None:
                            raise PlanError("the tile grid starts at a parameter")
                        s.span.append(Span(d, tiled[d], lb, lb + tiled[d] - 1))
                    else:
                        if lb is None or ub is None:
                            raise PlanError("an untiled dimension of run-time length")
                        s.span.append(Span(None, 0, lb, ub))
            else:
                s.span = self._requested(s, 'span')
                if s.span is None:
                    raise PlanError("%s is read nowhere" % s.name)
                for i in range(s.nd):
                    s.span[i] = self._clip(s, i, s.span[i])
        # stages of one phase with equal boxes share a sweep
        self.sweeps = []
        for ph in range(self.nphases):
            groups = {}
            for s in self.stages:
                if not s.inline and s.phase == ph:
                    groups.setdefault(tuple(sp.key() for sp in s.span), []).append(s)
            self.sweeps += [(ph, g) for g in groups.values()]
        # blocks, readers first (a stage's LDS rows hold all that its
        # readers' blocks touch)
        for s in self.stages:
            s.pspan = None
        for (ph, g) in reversed(self.sweeps):
            self._block(g)
        for s in self.stages:
            s.rspan = self._requested(s, 'pspan') if s is not a and not s.inline else None

    def _points(self, s):
        """Span of the points s is computed at."""
        return self._requested(s, 'pspan') if s.inline else s.pspan

    def _check_ref(self, s, r):
        """C's truncating division equals the floor division of the plan's
        maps on every coordinate that counts."""
        for arg in r.arguments:
            m = arg_map(arg, s.func.variables)
            if m.kind != 'var' or m.period == 1:
                continue
            lb = const_int(s.func.domain[m.dim].lowerBound)
            core = _strip_clamp(arg)
            core = Value.numericToValue(arg) if core is None else core[0]
            if lb is None or any(ceval_int(n, {s.func.variables[m.dim]: lb}) < 0
                                 for n in _divisors(core)[1]):
                # (an index like (x - 1) / 2 that only odd points take)
                raise PlanError("division of a negative coordinate")

    def _clip(self, s, i, sp):
        """A constant span cut to the domain and the hull of the Cases."""
        if sp.A:
            return sp
        lo, hi = const_int(s.func.domain[i].lowerBound), const_int(s.func.domain[i].upperBound)
        l, h = sp.lo, sp.hi
        if lo is not None:
            l = max(l, lo)
        if hi is not None:
            h = min(h, hi)
        los = [const_int(p.box[i][0]) if p.box[i][0] is not None else lo for p in s.parts]
        his = [const_int(p.box[i][1]) if p.box[i][1] is not None else hi for p in s.parts]
        if None not in los:
            l = max(l, min(los))
        if None not in his:
            h = min(h, max(his))
        if l > h:
            raise PlanError("%s: empty box" % s.name)
        return Span(None, 0, l, h)

    def _requested(self, s, which):
        """Hull of the points of s that its consumers' points (``span``:
        those that count; ``pspan``: all that are computed) read."""
        out = None
        for (c, part, r) in s.consumers:
            if any(self._part_span(c, part, j) is None for j in range(c.nd)):
                continue
            req = []
            for i, arg in enumerate(r.arguments):
                m = arg_map(arg, c.func.variables)
                if m.kind == 'const':
                    req.append(Span(None, 0, m.value, m.value))
                elif m.kind == 'var' and not (m.lows or m.highs):
                    sp = self._part_span(c, part, m.dim) if which == 'span' else self._points(c)[m.dim]
                    req.append(image(m, sp))
                else:
                    lo = const_int(s.func.domain[i].lowerBound)
                    hi = const_int(s.func.domain[i].upperBound)
                    if lo is None or hi is None:
                        raise PlanError("a data-dependent read of a tiled stage")
                    req.append(Span(None, 0, lo, hi))
            out = req if out is None else [x.hull(y) for x, y in zip(out, req)]
        return out

    def _block(self, members):
        """The per-thread block of a sweep: ``blk`` points per dimension,
        ``cnt`` blocks.

        Constant dimensions of up to 8 points are taken whole when points
        along them share reads (colours that all read alpha, intensity
        levels of one gray value) or differ in their Case; along rows and
        columns the block is a multiple of every parity (period 2 or 4)
        that an index or remainder of the stage uses; an index of another
        period is computed per point.  Among the sizes left,
        the smallest of an estimate is taken: (wavefronts of items, half of
        them rounded up to whole workgroup iterations) x (fixed cost + points
        x operations + distinct loads)."""
        threads = int(self.opts.get('threads', 256))
        s = members[0]
        nd = s.nd
        span = s.span
        blk = [1] * nd
        ext = [sp.ext for sp in span]
        req = [1] * nd
        maps = []
        nops = 4.0
        for m in members:
            stages = [m] + self._inline_closure(m)
            for (t, r) in self.closure_refs(m):
                ms = [arg_map(x, t.func.variables) for x in r.arguments]
                maps.append((t, r, ms))
                for x in ms:
                    if x.kind == 'var' and x.period in (2, 4):
                        req[x.dim] = max(req[x.dim], x.period)
            for t in stages:
                nops += sum(_nops(p.expr) for p in t.parts) / float(len(t.parts))
                for part in t.parts:
                    for (k, x) in _mods(part.expr, t.func.variables, least_values(t.func, part)):
                        if x in (2, 4):
                            req[k] = max(req[k], x)
        cd, rd = nd - 1, nd - 2
        if span[cd].A == 0 and ext[cd] <= 4 and nd >= 2:
            blk[cd] = ext[cd]
            cd, rd = nd - 2, nd - 3
        for i in range(nd):
            if i in (rd, cd) or span[i].A or ext[i] > 8 or blk[i] > 1:
                continue
            shares = any(not any(x.kind == '*' or (x.kind == 'var' and x.dim == i) for x in ms)
                         for (t, r, ms) in maps) or \
                any(p.box[i] != (None, None) for m in members for t in [m] + self._inline_closure(m)
                    for p in t.parts if len(t.parts) > 1)
            if shares:
                blk[i] = ext[i]
        for i in range(nd):
            # a tile that is no multiple of the parity changes it from tile
            # to tile: indices are then computed per point
            if span[i].A % req[i] or i not in (rd, cd):
                req[i] = 1
        whole = len(members)
        for x in blk:
            whole *= x
        best = None
        asked = (self.opts.get('box_blocks') or {}).get(s.name)
        if asked is not None:
            # (gpu option box_blocks: {first stage of a sweep: [U, V]})
            best = (None, [asked[0] if i == rd else asked[1] if i == cd else k
                           for i, k in enumerate(blk)])
        for U in ((1, 2, 4, 8) if rd >= 0 and best is None else (1,) if best is None else ()):
            for V in (1, 2, 4):
                if rd >= 0 and U % req[rd] or V % req[cd]:
                    continue
                if rd >= 0 and U > max(int(self.opts.get('box_rows', U)), req[rd]) and \
                        any(m.needs_lds for m in members):
                    continue
                least = (req[rd] if rd >= 0 else 1) * req[cd]
                if U * V > least and (whole * U * V > MAX_POINTS or
                                      (rd >= 0 and U > req[rd] and ext[rd] < 2 * U) or
                                      (V > req[cd] and ext[cd] < 4 * V)):
                    continue
                b = list(blk)
                b[cd] = V
                if rd >= 0:
                    b[rd] = U
                items = 1
                pts = 1
                for e, k in zip(ext, b):
                    items *= -(-e // k)
                    pts *= k
                c = 12.0 + pts * nops + self._loads(s, maps, b, V, cd)
                if any(m.liveout for m in members):
                    c += 3.0 * pts / V
                waves = 0.5 * (-(-items // 64)) + 0.5 * (-(-items // threads)) * (threads / 64.0)
                if best is None or (waves * c, -pts) < best[0]:
                    best = ((waves * c, -pts), b)
        if best is None:
            raise PlanError("no block holds every parity of %s" % s.name)
        for m in members:
            m.blk = list(best[1])
            m.base = [sp.lo for sp in span]
            m.cnt = [-(-e // k) for e, k in zip(ext, m.blk)]
            m.pspan = [Span(sp.d, sp.A, sp.lo, sp.lo + c * k - 1)
                       for sp, c, k in zip(span, m.cnt, m.blk)]

    def _inline_closure(self, s):
        out = []
        for (t, r) in self.closure_refs(s):
            if self.in_group(r.objectRef):
                p = self.stage_of(r.objectRef)
                if p.inline and p not in out:
                    out.append(p)
        return out

    def _loads(self, s, maps, blk, V, cd):
        """Estimated cost of a block's distinct loads."""
        import itertools
        total = 0.0
        pts = list(itertools.product(*[range(b) for b in blk]))
        runs = {}
        for (t, r, ms) in maps:
            if self.in_group(r.objectRef) and self.stage_of(r.objectRef).inline:
                continue
            dyn = any(m.kind == '*' or (m.kind == 'var' and blk[m.dim] % m.period and m.period > 1)
                      for m in ms)
            if dyn:
                # a sum per computed index and point; an index that varies
                # along one dimension only is computed once per row of it.
                # (A bilateral slice reads one grid row for 8 rows of pixels:
                # 8x1 points a thread share it, 4x2 compute it 4 times; on
                # 64x64 tiles 33.6 against 29.4 us for 2560x1536.)
                along = set(m.dim for m in ms if m.kind == 'var' and
                            m.period > 1 and blk[m.dim] % m.period)
                total += (3.0 + len(along) + any(m.kind == '*' for m in ms)) * len(pts)
                total += 3.0 * sum(blk[i] for i in along)
                continue
            seen = runs.setdefault((r.objectRef, tuple((m.kind, m.dim, m.slope) for m in ms)), set())
            for u in pts:
                seen.add(tuple(m.value if m.kind == 'const' else m.f(s.span[m.dim].lo + u[m.dim])
                               for m in ms))
        for key, seen in runs.items():
            # every distinct element costs its conversion and its share of
            # the memory pipe's width; LDS rows come in chunks of 2 or 4
            n = float(len(seen))
            if not self.in_group(key[0]):
                total += (5.0 if V < 4 else 6.0) * n
                continue
            last = key[1][-1] if key[1] else ('const', None, None)
            w = 1
            if last[0] == 'var' and last[1] == cd and last[2] * V >= 2:
                w = 4 if last[2] * V % 4 == 0 else 2
            chunks = set(x[:-1] + (x[-1] // w,) for x in seen)
            total += 2.0 * n + len(chunks) * (0.8 + 0.7 * w)
        return total

    # -- LDS -----------------------------------------------------------------------
    def _layout(self):
        """LDS rows: every point the stage computes and every point its
        readers' blocks touch; row starts and the stage's own blocks on
        16-byte boundaries.  Buffers are reused by phase (GroupPlan._storage's
        rule on these sizes)."""
        for s in self.stages:
            if not s.needs_lds:
                continue
            n = s.func.typ.nbytes()
            s.lspan = [x.hull(y) for x, y in zip(s.pspan, s.rspan)]
            al = max(1, 16 // n)
            last = s.lspan[-1]
            if last.ext >= 4:
                lo = s.base[-1] - -(-(s.base[-1] - last.lo) // al) * al
                s.lspan[-1] = Span(last.d, last.A, lo, last.hi)
            s.lext = [sp.ext for sp in s.lspan]
            if last.ext >= 4:
                s.lext[-1] = -(-s.lext[-1] // al) * al
            s.vread = True          # (16 bytes of slack after the last row)
        self._storage()

    def lds_ext(self, s):
        return s.lext
